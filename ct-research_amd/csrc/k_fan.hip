// k_fan.hip - fan-beam pixel-driven kernels for gfx950: the reference
// backprojection (linear sample x pixel chord), the exact adjoint of the
// Siddon fan projector, and the flat / equiangular FBP backprojection.
// The views of a pixel are split over the wavefronts of its block where one
// thread per pixel would leave the chip waiting (the reference launches one
// kernel per view, BackprojectionFan2D.cu:243-314).
#include "ctr_internal.h"

#include <cmath>

namespace ctr {
namespace {

// Reference fan backprojection (BackprojectionFan2D.cu:7-116).
__global__ __launch_bounds__(256) void k_fan_bp_ref(const float *__restrict__ proj, float *__restrict__ img, FanParams P)
{
    const int i = blockIdx.x * 16 + (threadIdx.x & 15), j = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (i >= P.nt || j >= P.ns) return;
    const float x = ((float)i + 0.5f) * P.rt - P.ct, y = ((float)j + 0.5f) * P.rs - P.cs;
    float acc = 0.0f;
    for (int b = 0; b < P.nb; ++b) {
        float val = 0.0f, chord;
        const float *r = proj + (size_t)b * P.np;
        if (!P.quirks) {
            const float sb = (float)P.view[4 * b + 0], cb = (float)P.view[4 * b + 1];
            const float u = x * cb + y * sb, s = -x * sb + y * cb;
            const float U = (P.D - s) / P.D;
            const float uu = fmaf(u / U, P.u_scale, P.u_off);
            if (uu >= 0.0f && uu < P.umax) {
                const int iu = min((int)floorf(uu), (int)P.umax - 1);
                const float fu = uu - (float)iu;
                val = fmaf(fu, r[iu + 1] - r[iu], r[iu]);
            }
            // the line from the source through the pixel centre: chord = 2 |d| min(h/|d_axis|)
            const float dx = x + P.ct - (float)P.view[4 * b + 2], dy = y + P.cs - (float)P.view[4 * b + 3];
            chord = 2.0f * sqrtf(dx * dx + dy * dy) * fminf(0.5f * P.rt / fabsf(dx), 0.5f * P.rs / fabsf(dy));
        } else {
            // the reference's arithmetic in FP64 (its face test is discontinuous, so
            // rounding must follow it): entry face tested against 0 instead of the
            // pixel's low edge (:95-101), distance taken to the ray's far end point (:109)
            const double Db = P.D, st = P.view[4 * b + 2], ss = P.view[4 * b + 3];
            const double sbd = P.view[4 * b + 0], cbd = P.view[4 * b + 1];
            const double ct = P.ct_d, cs = P.cs_d;
            const double xd = ((double)i + 0.5) * P.rt_d - ct, yd = ((double)j + 0.5) * P.rs_d - cs;
            const double ud = xd * cbd + yd * sbd, sd = -xd * sbd + yd * cbd;
            const double pd = ud / ((Db - sd) / Db);
            const double uu = pd * P.u_scale_d + P.u_off_d;
            if (uu >= 0.0 && uu < (double)P.umax) {
                const int iu = min((int)floor(uu), (int)P.umax - 1);
                const double fu = uu - (double)iu;
                val = (float)((1.0 - fu) * (double)r[iu] + fu * (double)r[iu + 1]);
            }
            const double th = atan(pd / Db), Smax = 2.0 * Db;
            const double te = ct + Smax * sin(th) * cbd - (Db - Smax * cos(th)) * sbd;
            const double se = cs + Smax * sin(th) * sbd + (Db - Smax * cos(th)) * cbd;
            double t2s = (se - ss) / ((te - st) == 0.0 ? 1e-15 : (te - st));
            double s2t = (te - st) / ((se - ss) == 0.0 ? 1e-15 : (se - ss));
            t2s = fmin(fmax(t2s, -1e16), 1e16);
            s2t = fmin(fmax(s2t, -1e16), 1e16);
            const double tlo = (double)i * P.rt_d, thi = (double)(i + 1) * P.rt_d;
            const double slo = (double)j * P.rs_d, shi = (double)(j + 1) * P.rs_d;
            const double tlo_s = ss + (tlo - st) * t2s, slo_t = st + (slo - ss) * s2t;
            double T1, S1;
            if (tlo_s >= 0.0 && tlo_s <= shi) {
                T1 = tlo;
                S1 = tlo_s;
            } else if (slo_t >= 0.0 && slo_t <= thi) {
                T1 = slo_t;
                S1 = slo;
            } else {
                continue;
            }
            chord = (float)(2.0 * sqrt((T1 - te) * (T1 - te) + (S1 - se) * (S1 - se)));
        }
        acc = fmaf(val, chord, acc);
    }
    const size_t o = (size_t)j * P.nt + i;
    img[o] = P.accumulate ? img[o] + acc : acc;
}

// ---------------------------------------------------------------------------
// Exact adjoint of the fan Siddon projector, for any monotone detector.  Per
// pixel and view the candidate rays are the bins whose positions fall inside
// the projection of the pixel's square.  The ray S + lam (a, b) through bin p,
// a = p cos + D sin, b = p sin - D cos, meets the pixel for lam in the
// intersection of its t and s slabs.  The slab parameters are measured from
// the source, D away, so they are formed in FP64 with the FP64 bin positions
// of the forward projector.  The records n/a, n/b (n = |(a, b)|, so that lam is
// a length) are a table of the geometry; a geometry whose table would be too
// large forms them as it goes.
// ---------------------------------------------------------------------------
// n/a and n/b; a component of exactly 0 gives a finite 1e300, whose slab
// interval holds every positive lam when the source lies in the slab and none
// otherwise.
__device__ __forceinline__ double2 fan_ray(double sb, double cb, double p, double D)
{
    const double a = p * cb + D * sb, b = p * sb - D * cb, n = sqrt(p * p + D * D);
    return make_double2(a != 0.0 ? n / a : 1e300, b != 0.0 ? n / b : 1e300);
}

__global__ __launch_bounds__(256) void k_fan_ray_table(FanParams P, double2 *__restrict__ out)
{
    const size_t n = (size_t)P.nb * P.np;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (size_t)gridDim.x * 256) {
        const size_t b = e / P.np;
        out[e] = fan_ray(P.view[4 * b], P.view[4 * b + 1], P.pdbl[e - b * P.np], (double)P.D);
    }
}

// Length of the ray in the pixel whose faces lie at t0, t1 and s0, s1 from the source.
__device__ __forceinline__ float fan_length(double2 ray, double t0, double t1, double s0, double s1)
{
    const double a0 = t0 * ray.x, a1 = t1 * ray.x, b0 = s0 * ray.y, b1 = s1 * ray.y;
    const double lo = fmax(fmin(a0, a1), fmin(b0, b1)), hi = fmin(fmax(a0, a1), fmax(b0, b1));
    return fmaxf((float)(hi - lo), 0.0f);
}

// Smallest / largest int of a wavefront by lane permutations (quad, half row,
// row, then the rows' last lanes into the next rows): no LDS round trips.
template <int CTRL>
__device__ __forceinline__ int lane_perm(int v)
{
    return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ int wave_min_i(int v)
{
    v = min(v, lane_perm<0xB1>(v));
    v = min(v, lane_perm<0x4E>(v));
    v = min(v, lane_perm<0x141>(v));
    v = min(v, lane_perm<0x140>(v));
    v = min(v, lane_perm<0x142>(v));
    v = min(v, lane_perm<0x143>(v));
    return __builtin_amdgcn_readlane(v, 63);
}

// Orders a wave's own LDS accesses (they execute in issue order).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kFanWaves = 8;     // views of a round, at most: one per wave of the block
constexpr int kFanStage = 64;    // rays of a view staged per wave
constexpr int kFanSlots = 6;     // lengths a pixel keeps per view (a pixel of two bins' width meets 5 at most)

// A block owns 8 x 8 pixels.  In a round its 8 waves form the lengths of 8
// views, one wave per view and one lane per pixel, and leave them in LDS;
// after the round's barrier one wave (each in its turn) adds length times
// sample to the pixels' sums, view after view and bin after bin, while the
// others form the next round's.  The sum of a pixel thus runs through the same
// float fma chain as with one thread over all views (a residual history of
// SIRT depends on it at 1e-8), and the work of forming the lengths has 8 waves
// per tile: a 256^2 image gives the chip 32 waves per CU instead of 4.
//
// Per view a wave finds each pixel's shadow on the detector (its centre and
// half width, widened by a margin for the float arithmetic), looks the bins up
// in a table of bin indices over the detector, and stages the records and
// samples of the tile's rays into LDS.  A view in which a pixel meets more
// than kFanSlots rays, or the tile more than kFanStage, is summed from the
// table by the adding wave.
//
// 256^2 pixels, 360 views, 512 equiangular bins: 1193 us with one thread per
// pixel, two binary searches per view and four FP64 divisions and a root per
// ray; 200 us now, VALU issue (about 200 instructions per wave and view: 50 to
// find the bins, 75 for the lengths, 35 to add).
//
// A block has W waves: as many as views, rounded up to a power of two, where that
// is less than 8 (a single view or a few of an ordered subset: the others would
// only hold room).  One view of 2048^2 pixels, 1024 bins: 51 us with one thread
// per pixel, 109 us by blocks of 8 waves, 27 us by one; two views 89 / 127 / 49
// us.
template <bool TABLE, int W>
__global__ __launch_bounds__(64 * W, 8) void k_fan_adjoint(const float *__restrict__ proj, float *__restrict__ img,
                                                          FanParams P, SirtUpdate U, int sirt, int ones)
{
    __shared__ double2 rays[W][kFanStage];
    __shared__ float ys[2][W][kFanStage];
    __shared__ float slot[2][W][kFanSlots][64];
    __shared__ unsigned char first[2][W][64];   // the pixel's first ray in ys
    __shared__ int count[2][W];   // slots in use, -1: a view for the adding wave
    __shared__ float sum[64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int i = blockIdx.x * 8 + (lane & 7), j = blockIdx.y * 8 + (lane >> 3);
    const bool in = i < P.nt && j < P.ns;
    const double tlo = (double)i * P.rt_d, thi = tlo + P.rt_d, slo = (double)j * P.rs_d, shi = slo + P.rs_d;
    const float x = ((float)i + 0.5f) * P.rt - P.ct, y = ((float)j + 0.5f) * P.rs - P.cs;
    const float hx = 0.5f * P.rt, hy = 0.5f * P.rs;
    const float cell_max = (float)(P.lut_n - 1);
    if (wave == 0) sum[lane] = 0.0f;

    // first and last candidate bin of this lane's pixel in view b
    auto bins = [&](int b, int &c0, int &c1) {
        const float sb = (float)P.view[4 * (size_t)b], cb = (float)P.view[4 * (size_t)b + 1];
        // a corner (+-hx, +-hy) moves the projection D u / ds by
        // D (du ds + u dv) / (ds (ds - dv))
        const float u = fmaf(x, cb, y * sb), ds = P.D - fmaf(-x, sb, y * cb);
        const float far = fmaf(hx, fabsf(fmaf(cb, ds, -u * sb)), hy * fabsf(fmaf(sb, ds, u * cb)));
        const float near = ds - fmaf(hx, fabsf(sb), hy * fabsf(cb));
        const float q = P.D * __builtin_amdgcn_rcpf(ds), pc = u * q;
        const float dp = far * q * __builtin_amdgcn_rcpf(near);
        const float eu = fmaf(1e-5f, fabsf(pc) + dp, P.lut_eps);
        float lo = pc - dp - eu, hi = pc + dp + eu;
        if (!(near > 1e-4f * P.D)) {   // a pixel next to the source orbit: every ray
            lo = -kInf;
            hi = kInf;
        }
        const int k0 = (int)__builtin_amdgcn_fmed3f((lo - P.lut_lo) * P.lut_scale, 0.0f, cell_max);
        const int k1 = (int)__builtin_amdgcn_fmed3f((hi - P.lut_lo) * P.lut_scale, 0.0f, cell_max);
        const int f = P.lut[k0], l = P.lut[k1 + 1];   // in ascending position
        c0 = P.asc ? f : P.np - l;
        c1 = (P.asc ? l : P.np - f) - 1;
        if (!in) {
            c0 = 0x7fffffff;
            c1 = -1;
        }
    };
    auto record = [&](int b, int c) {
        return TABLE ? P.rays[(size_t)b * P.np + c]
                     : fan_ray(P.view[4 * (size_t)b], P.view[4 * (size_t)b + 1], P.pdbl[c], (double)P.D);
    };
    // view b, whose bins c0 .. c1 are known, into the slots of buffer h; the
    // bins of the wave's next view are looked up behind the records' loads
    int c0 = 0x7fffffff, c1 = -1;
    auto form = [&](int b, int h) {
        const int cmin = wave_min_i(c0);
        const bool fits = __ballot(c1 - cmin >= kFanStage || c1 - c0 >= kFanSlots) == 0;
        int n = 0;
        while (n < kFanSlots && __ballot(c1 - c0 >= n)) ++n;
        if (lane == 0) count[h][wave] = fits ? n : -1;
        const int cl = min(cmin + lane, P.np - 1);
        const double2 ray = record(b, cl);
        const float yv = ones ? 1.0f : proj[(size_t)b * P.np + cl];
        const int rel = in ? c0 - cmin : 0, mine = in ? c1 - c0 : -1;
        if (b + W < P.nb) bins(b + W, c0, c1);
        if (!fits) return;
        rays[wave][lane] = ray;
        ys[h][wave][lane] = yv;
        first[h][wave][lane] = (unsigned char)rel;
        wave_sync();
        const double st = P.view[4 * (size_t)b + 2], ss = P.view[4 * (size_t)b + 3];
        const double t0 = tlo - st, t1 = thi - st, s0 = slo - ss, s1 = shi - ss;
        // rays of one direction, as in all views but those along an axis, enter
        // every pixel through the same two faces: no sorting of the parameters
        const unsigned long long px = __ballot(ray.x > 0.0), py = __ballot(ray.y > 0.0);
        if ((px == 0 || px == ~0ull) && (py == 0 || py == ~0ull)) {
            const double tn = px ? t0 : t1, tf = px ? t1 : t0, sn = py ? s0 : s1, sf = py ? s1 : s0;
            for (int k = 0; k < n; ++k) {
                const double2 q = rays[wave][(rel + k) & (kFanStage - 1)];
                const double lo = fmax(tn * q.x, sn * q.y), hi = fmin(tf * q.x, sf * q.y);
                slot[h][wave][k][lane] = k <= mine ? fmaxf((float)(hi - lo), 0.0f) : 0.0f;
            }
        } else {
            for (int k = 0; k < n; ++k) {
                const float len = fan_length(rays[wave][(rel + k) & (kFanStage - 1)], t0, t1, s0, s1);
                slot[h][wave][k][lane] = k <= mine ? len : 0.0f;
            }
        }
        wave_sync();   // the next view's records go where these were read
    };
    // a length of 0 adds nothing, whatever the sample holds
    auto add = [](float len, float yv, float acc) { return len != 0.0f ? fmaf(len, yv, acc) : acc; };

    const int rounds = (P.nb + W - 1) / W;
    if (wave < P.nb) {
        bins(wave, c0, c1);
        form(wave, 0);
    }
    for (int r = 0; r < rounds; ++r) {
        const int h = r & 1, next = (r + 1) * W + wave;
        __syncthreads();
        if (r % W == wave) {
            float acc = sum[lane];
            for (int w = 0; w < W && r * W + w < P.nb; ++w) {
                const int n = __builtin_amdgcn_readfirstlane(count[h][w]);
                if (n >= 0) {
                    const int rel = first[h][w][lane];
                    for (int k = 0; k < n; ++k)
                        acc = add(slot[h][w][k][lane], ys[h][w][(rel + k) & (kFanStage - 1)], acc);
                } else {
                    const int b = r * W + w;
                    int c0, c1;
                    bins(b, c0, c1);
                    const double st = P.view[4 * (size_t)b + 2], ss = P.view[4 * (size_t)b + 3];
                    for (int c = c0; c <= c1; ++c)
                        acc = add(fan_length(record(b, c), tlo - st, thi - st, slo - ss, shi - ss),
                                  ones ? 1.0f : proj[(size_t)b * P.np + c], acc);
                }
            }
            sum[lane] = acc;
        }
        if (next < P.nb) form(next, h ^ 1);
    }
    __syncthreads();
    if (wave != 0 || !in) return;
    const float acc = sum[lane];
    const size_t o = (size_t)j * P.nt + i;
    if (sirt) {
        const float xn = fmaf(U.lambda * U.vinv[o], acc, U.x[o]);
        U.x[o] = fminf(fmaxf(xn, U.lo), U.hi);
    } else {
        img[o] = P.accumulate ? img[o] + acc : acc;
    }
}

// The FBP backprojections sum every view at every pixel: little memory (the
// filtered views stay in L2), so they are bound by vector issue once enough
// wavefronts are in flight.  A block of W wavefronts covers one tile of
// pixels; wavefront w sums views w, w + W, ..., and the W sums are added in
// order.  With a thread per pixel (all views in one chain, four wavefronts per
// CU at 256^2) issue waited on each view's loads and divisions.
constexpr int kBpWaves = 8;

template <int NP>
__device__ __forceinline__ void add_waves(float (&acc)[NP], float (*part)[NP][64], int wave, int lane)
{
#pragma unroll
    for (int k = 0; k < NP; ++k) part[wave][k][lane] = acc[k];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int w = 1; w < kBpWaves; ++w)
#pragma unroll
        for (int k = 0; k < NP; ++k) acc[k] += part[w][k][lane];
}

// 1 / v to within an ulp (v normal)
__device__ __forceinline__ float reciprocal(float v)
{
    const float r = __builtin_amdgcn_rcpf(v);
    return fmaf(fmaf(-v, r, 1.0f), r, r);
}

// Fan FBP backprojection.
//   flat (FBPfan.cu:45-96): sum_b lerp(q)(p/U) / U^2 * dbeta, U = (D - s)/D
//   equiangular (FanProjection.m:299-324): sum_b lerp(q)(gamma) / L^2 * dbeta,
//   gamma = atan2(u, D - s), L^2 = u^2 + (D - s)^2
// 8 x 8 pixels a block.  Where every lane's |u| < (D - s)/2, as inside any
// usual fan, gamma is fan_atan(u / (D - s)); atan2f else.  360 views, 256^2, equiangular: 160 us for a
// thread per pixel, 43 us by eight wavefronts, 30 us with the shorter
// angle and reciprocals.
template <bool EQUIANGULAR>
__global__ __launch_bounds__(64 * kBpWaves, 8) void k_fan_fbp_bp(const float *__restrict__ filt,
                                                                 float *__restrict__ img, FanParams P)
{
    __shared__ float part[kBpWaves][1][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = blockIdx.x * 8 + (lane & 7), j = blockIdx.y * 8 + (lane >> 3);
    const bool in = i < P.nt && j < P.ns;
    const float x = ((float)i + 0.5f) * P.rt - P.ct, y = ((float)j + 0.5f) * P.rs - P.cs;
    float acc[1] = {0.0f};
    for (int b = wave; b < P.nb; b += kBpWaves) {
        const float sb = (float)P.view[4 * b + 0], cb = (float)P.view[4 * b + 1];
        const float u = x * cb + y * sb, s = -x * sb + y * cb, w = P.D - s;
        float pos, weight;
        bool hit;
        if (!EQUIANGULAR) {
            // p / U = D u / w, 1 / U^2 = (D / w)^2
            const float r = reciprocal(w), q0 = u * r, q = fmaf(fmaf(-q0, w, u), r, q0), m = P.D * r;
            pos = fmaf(P.D * q, P.u_scale, P.u_off);
            weight = m * m;
            hit = pos >= 0.0f && pos < P.umax;
        } else {
            float g;
            if (__all(!in || fabsf(u) < kFanAtanMax * fabsf(w))) {
                const float v = fabsf(w), r = __builtin_amdgcn_rcpf(v), q0 = u * r;
                g = fan_atan(fmaf(fmaf(-q0, v, u), r, q0));
            } else {
                g = atan2f(u, fabsf(w));
            }
            pos = (g - P.g0) * P.g_scale;
            weight = reciprocal(fmaf(u, u, w * w));
            hit = pos >= 0.0f && pos < P.gmax;
        }
        if (in && hit) {
            // linear interpolation, in the equiangular case in gamma
            // (FanProjection.m:93-98) on the uniform angle grid
            const int k = min((int)pos, (int)(EQUIANGULAR ? P.gmax : P.umax) - 1);
            const float *r = filt + (size_t)b * P.np;
            const float f = pos - (float)k;
            acc[0] = fmaf(fmaf(f, r[k + 1] - r[k], r[k]), weight, acc[0]);
        }
    }
    add_waves(acc, part, wave, lane);
    if (wave != 0 || !in) return;
    const size_t o = (size_t)j * P.nt + i;
    img[o] = P.accumulate ? img[o] + acc[0] * P.dbeta : acc[0] * P.dbeta;
}

// Parallel-beam FBP backprojection (FBPparallel.cu:41-89; the reference
// launches one kernel per view and adds into the image).  16 x 16 pixels a
// block, four to a lane.  The tile's shadow on the detector is at most 16
// diagonals: where that is less than 57 bins (STAGED) lane l of a wavefront
// loads bin c0 + l of the shadow and the pixels take their two bins from those
// lanes (ds_bpermute); the bins of lanes 62 and 63 are zero for the pixels that
// miss the detector.  Gathers from memory otherwise.
// 360 views, 512^2, 730 bins of 1.1 pixels: 115 us for a thread per
// pixel, 66 us by eight wavefronts with gathers (bound by the texture unit, one
// gather of two bins per 64 pixels), 46 us with the shadow in registers.
constexpr int kParTile = 16, kParSpan = 57;
template <bool STAGED>
__global__ __launch_bounds__(64 * kBpWaves, 8) void k_par_fbp_bp(const float *__restrict__ filt,
                                                                 float *__restrict__ img, ParBpParams P)
{
    __shared__ float part[kBpWaves][4][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i0 = blockIdx.x * kParTile, j0 = blockIdx.y * kParTile;
    float x[2], y[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        x[k] = ((float)(i0 + (lane & 7) + 8 * k) + 0.5f) * P.rt - P.ct;
        y[k] = ((float)(j0 + (lane >> 3) + 8 * k) + 0.5f) * P.rs - P.cs;
    }
    const float xm = ((float)i0 + 0.5f * kParTile) * P.rt - P.ct, ym = ((float)j0 + 0.5f * kParTile) * P.rs - P.cs;
    const float hx = 0.5f * (kParTile - 1) * P.rt * fabsf(P.u_scale), hy = 0.5f * (kParTile - 1) * P.rs * fabsf(P.u_scale);
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int b = wave; b < P.nb; b += kBpWaves) {
        const float sb = P.view[2 * b], cb = P.view[2 * b + 1];
        const float *row = filt + (size_t)b * P.np;
        float bin = 0.0f;
        int c0 = 0;
        if (STAGED) {
            const float um = fmaf(fmaf(xm, cb, ym * sb), P.u_scale, P.u_off);
            c0 = __builtin_amdgcn_readfirstlane((int)floorf(um - fmaf(hx, fabsf(cb), hy * fabsf(sb)))) - 1;
            const int c = c0 + lane;
            if (c >= 0 && c < P.np && lane < 62) bin = row[c];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float u = fmaf(fmaf(x[k & 1], cb, y[k >> 1] * sb), P.u_scale, P.u_off);
            const float fl = floorf(u);
            const int iu = (int)fl;
            const bool hit = u >= 0.0f && u < P.umax;
            const float f = STAGED || hit ? u - fl : 0.0f;   // u is finite in a staged tile
            float a = 0.0f, d = 0.0f;
            if (STAGED) {
                const int at = (hit ? iu - c0 : 62) * 4;
                a = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(at, __builtin_bit_cast(int, bin)));
                d = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(at + 4, __builtin_bit_cast(int, bin)));
            } else if (hit) {
                a = row[min(iu, P.np - 2)];
                d = row[min(iu, P.np - 2) + 1];
            }
            acc[k] += fmaf(f, d - a, a);
        }
    }
    add_waves(acc, part, wave, lane);
    if (wave != 0) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int i = i0 + (lane & 7) + 8 * (k & 1), j = j0 + (lane >> 3) + 8 * (k >> 1);
        if (i >= P.nt || j >= P.ns) continue;
        const size_t o = (size_t)j * P.nt + i;
        img[o] = P.accumulate ? img[o] + acc[k] * P.dtheta : acc[k] * P.dtheta;
    }
}

dim3 pix_grid(const FanParams &P) { return dim3((P.nt + 15) / 16, (P.ns + 15) / 16); }

}  // namespace

hipError_t launch_fan_bp_ref(const FanParams &P, const float *proj, float *img, hipStream_t st)
{
    hipLaunchKernelGGL(k_fan_bp_ref, pix_grid(P), dim3(256), 0, st, proj, img, P);
    return hipGetLastError();
}

hipError_t launch_fan_ray_table(const FanParams &P, double2 *rays, hipStream_t st)
{
    const size_t n = (size_t)P.nb * P.np, blocks = (n + 255) / 256;
    hipLaunchKernelGGL(k_fan_ray_table, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(256), 0, st, P, rays);
    return hipGetLastError();
}

template <int W>
static void launch_fan_adjoint_waves(const FanParams &P, const float *proj, float *img, const SirtUpdate &U, int sirt,
                                     int ones_input, hipStream_t st)
{
    const dim3 grid((P.nt + 7) / 8, (P.ns + 7) / 8), block(64 * W);
    if (P.rays) hipLaunchKernelGGL((k_fan_adjoint<true, W>), grid, block, 0, st, proj, img, P, U, sirt, ones_input);
    else hipLaunchKernelGGL((k_fan_adjoint<false, W>), grid, block, 0, st, proj, img, P, U, sirt, ones_input);
}

hipError_t launch_fan_adjoint(const FanParams &P, const float *proj, float *img, const SirtUpdate *upd, int ones_input,
                              hipStream_t st)
{
    SirtUpdate U = {};
    int sirt = 0;
    if (upd) {
        U = *upd;
        sirt = 1;
    }
    if (P.nb > 4) launch_fan_adjoint_waves<kFanWaves>(P, proj, img, U, sirt, ones_input, st);
    else if (P.nb > 2) launch_fan_adjoint_waves<4>(P, proj, img, U, sirt, ones_input, st);
    else if (P.nb > 1) launch_fan_adjoint_waves<2>(P, proj, img, U, sirt, ones_input, st);
    else launch_fan_adjoint_waves<1>(P, proj, img, U, sirt, ones_input, st);
    return hipGetLastError();
}

// Exact adjoint of the parallel Siddon projector.  Per pixel and view the
// candidate rays are the bins inside the pixel's shadow on the detector.  A
// ray at signed distance dl (along n = (cos, sin)) from the pixel centre,
// parameterised by mu along (-sin, cos) from the foot of the centre, has
// offsets (dl cos - mu sin, dl sin + mu cos) from the centre; its length in
// the pixel is the mu interval where both stay within the half pitches.  The
// centre's detector coordinate is formed in FP64 so that dl keeps its
// precision far from the rotation centre.
__global__ __launch_bounds__(256) void k_par_adjoint(const float *__restrict__ proj, float *__restrict__ img,
                                                     ParBpParams P, SirtUpdate U, int sirt, int ones)
{
    const int i = blockIdx.x * 16 + (threadIdx.x & 15), j = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (i >= P.nt || j >= P.ns) return;
    const double px = ((double)i + 0.5) * P.rt_d - P.ct_d, py = ((double)j + 0.5) * P.rs_d - P.cs_d;
    const float hx = 0.5f * P.rt, hy = 0.5f * P.rs;
    float acc = 0.0f;
    for (int b = 0; b < P.nb; ++b) {
        const double sbd = P.view_d[4 * b + 0], cbd = P.view_d[4 * b + 1];
        const float sb = (float)sbd, cb = (float)cbd;
        const double uc = fma(px, cbd, py * sbd);
        const float reach = fmaf(fabsf(cb), hx, fabsf(sb) * hy);
        float u0 = fmaf((float)uc - reach, P.u_scale, P.u_off), u1 = fmaf((float)uc + reach, P.u_scale, P.u_off);
        const float ulo = fminf(u0, u1), uhi = fmaxf(u0, u1);
        const float eu = 1e-3f + 4e-6f * fmaxf(fabsf(ulo), fabsf(uhi));
        const int c0 = max((int)ceilf(fminf(fmaxf(ulo - eu, -1.0f), (float)P.np)), 0);
        const int c1 = min((int)floorf(fminf(uhi + eu, (float)P.np)), P.np - 1);
        const float *r = proj + (size_t)b * P.np;
        for (int c = c0; c <= c1; ++c) {
            const float dl = (float)(P.t_d[c] - uc);
            const float ox = dl * cb, oy = dl * sb;
            float lo = -kInf, hi = kInf;
            if (sb != 0.0f) {
                const float inv = 1.0f / sb;
                const float l1 = (ox - hx) * inv, l2 = (ox + hx) * inv;
                lo = fmaxf(lo, fminf(l1, l2));
                hi = fminf(hi, fmaxf(l1, l2));
            } else if (!(ox >= -hx && ox < hx)) {
                continue;
            }
            if (cb != 0.0f) {
                const float inv = 1.0f / cb;
                const float l1 = (-hy - oy) * inv, l2 = (hy - oy) * inv;
                lo = fmaxf(lo, fminf(l1, l2));
                hi = fminf(hi, fmaxf(l1, l2));
            } else if (!(oy >= -hy && oy < hy)) {
                continue;
            }
            acc = fmaf(fmaxf(hi - lo, 0.0f), ones ? 1.0f : r[c], acc);
        }
    }
    const size_t o = (size_t)j * P.nt + i;
    if (sirt) {
        const float xn = fmaf(U.lambda * U.vinv[o], acc, U.x[o]);
        U.x[o] = fminf(fmaxf(xn, U.lo), U.hi);
    } else {
        img[o] = P.accumulate ? img[o] + acc : acc;
    }
}

hipError_t launch_par_fbp_bp(const ParBpParams &P, const float *filt, float *img, hipStream_t st)
{
    const dim3 grid((P.nt + kParTile - 1) / kParTile, (P.ns + kParTile - 1) / kParTile), block(64 * kBpWaves);
    // the shadow of a tile in bins, and the largest detector coordinate of a
    // pixel: below 2^18 the coordinates of one tile agree to far less than the
    // bin that the staged window has to spare on either side
    const double scale = std::fabs((double)P.u_scale), ext = kParTile - 1;
    const double span = std::hypot(ext * P.rt, ext * P.rs) * scale;
    const double far = (std::fabs(P.ct_d) + P.nt * P.rt_d + std::fabs(P.cs_d) + P.ns * P.rs_d) * scale + std::fabs(P.u_off);
    if (span < kParSpan && far < 262144.0)
        hipLaunchKernelGGL((k_par_fbp_bp<true>), grid, block, 0, st, filt, img, P);
    else
        hipLaunchKernelGGL((k_par_fbp_bp<false>), grid, block, 0, st, filt, img, P);
    return hipGetLastError();
}

hipError_t launch_par_adjoint(const ParBpParams &P, const float *proj, float *img, const SirtUpdate *U,
                              int ones_input, hipStream_t st)
{
    SirtUpdate u{};
    if (U) u = *U;
    hipLaunchKernelGGL(k_par_adjoint, dim3((P.nt + 15) / 16, (P.ns + 15) / 16), dim3(256), 0, st, proj, img, P, u,
                       U ? 1 : 0, ones_input);
    return hipGetLastError();
}

hipError_t launch_fan_fbp_bp(const FanParams &P, const float *filt, float *img, hipStream_t st)
{
    const dim3 grid((P.nt + 7) / 8, (P.ns + 7) / 8), block(64 * kBpWaves);
    if (P.equiangular) hipLaunchKernelGGL((k_fan_fbp_bp<true>), grid, block, 0, st, filt, img, P);
    else hipLaunchKernelGGL((k_fan_fbp_bp<false>), grid, block, 0, st, filt, img, P);
    return hipGetLastError();
}

}  // namespace ctr
