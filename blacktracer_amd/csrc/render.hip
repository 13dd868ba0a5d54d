// render.hip -- the per-pixel render pass (Path B): the drop-in for the
// G == 1 frame of cudaPrep (MakeImageKernel.cu:1402-1529).
//
// Stages, on the context stream but for what runs beside the star pass:
//   pix_interp   per pixel corner: quadtree descent of the dense grid and
//                bicubic Hermite interpolation of the celestial angle
//                (pixInterpolation, interpolatePix, kernel.cuh:736-968)
//   bh_area      shadow flag and celestial solid angle per pixel
//                (findBlackPixels + findArea)
//   smooth_h/v   box-filtered solid angle (smoothAreaH/V)
//   star pass    per pixel: candidate stars, point-in-quad, sub-pixel
//                position, blackbody colour and the Gaussian taps
//                (distortStarMap), a pixel's taps side by side: star_scan and
//                star_wide sort the pixels by their work, star_assign and
//                star_heads prepare the chunks of those with many candidates,
//                star_map_chunk and star_chunk_reduce trace them, star_few
//                and star_map_odd the others with a star inside
//   star_sum     gather of the neighbours' taps + makePix
//   env_map      summed-area sky sampling, lensing and redshift
//                (distortEnvironmentMap); env_map_group and env_map_heavy
//                for footprints of many sky columns
//   composite    addStarsAndBackground
// Pixel (i, j) is processed by thread x = j, y = i so that a wavefront
// (16 x 4 pixels of a 16 x 16 block) reads consecutive row addresses.
// Compiled with -ffp-contract=off: results equal the CPU oracle bit for bit.
#include <cmath>

#include "bt_render.h"
#include "render_dev.h"

namespace bt {
namespace {

using namespace rdr;

__constant__ int kTempRGB[1173] = {
#include "blackbody_rgb.inc"
};

struct Cam7 {
    float v[7];
    const float* colours;    // star_colours table, 391 x 6 floats
    const float* pix_area;   // per pixel: camera-sky solid angle of its view quad
};

__device__ __forceinline__ F2 gload(const float* grid, int GN, int GM, int i, int j) {
    if ((unsigned)i >= (unsigned)GN || (unsigned)j >= (unsigned)GM) return F2{-2.f, -2.f};
    const float2 v = reinterpret_cast<const float2*>(grid)[(size_t)i * GM + j];
    return F2{v.x, v.y};
}

struct GridV {
    const float* g;
    int GN, GM;
    float inv;   // 1 / GM for a power of two, else 0
    __device__ __forceinline__ F2 at(int i, int j) const { return gload(g, GN, GM, i, j); }
};

// kernel.cuh:774-788
__device__ F2 interpolate_linear(float percDown, float percRight, const F2* c) {
    float phi[4] = {c[0].y, c[1].y, c[2].y, c[3].y};
    float theta[4] = {c[0].x, c[1].x, c[2].x, c[3].x};
    pi_check(phi, 0.2f);
    float leftT = theta[0] + percDown * (theta[2] - theta[0]);
    float leftP = phi[0] + percDown * (phi[2] - phi[0]);
    float rightT = theta[1] + percDown * (theta[3] - theta[1]);
    float rightP = phi[1] + percDown * (phi[3] - phi[1]);
    float upT = theta[0] + percRight * (theta[1] - theta[0]);
    float upP = phi[0] + percRight * (phi[1] - phi[0]);
    float downT = theta[2] + percRight * (theta[3] - theta[2]);
    float downP = phi[2] + percRight * (phi[3] - phi[2]);
    return intersection(upT, upP, downT, downP, leftT, leftP, rightT, rightP);
}

// The reference's findPoint may recurse once into interpolateHermite
// (count 0 -> 1) and never deeper; the two levels are written out here.
__device__ __attribute__((noinline)) F2 interpolate_hermite_l1(GridV g, int i, int j, int gap, F2 c0, F2 c1, F2 c2, F2 c3);

// kernel.cuh:817-889 for recursion depth `count`, for a point (i, j) that the
// grid does not hold.  Out of line: most points are held, and the eight
// copies of this in every interpolation were larger than the instruction
// cache.
template <int COUNT>
__device__ __attribute__((noinline)) F2 find_missing(GridV g, int i, int j, int offver, int offhor, int gap) {
    const int GM = g.GM, GN = g.GN;
    int j2 = wrap_col(j + offhor * gap + GM, GM);
    int i2 = i + offver * gap;
    F2 ij2 = g.at(i2, j2);
    if (ij2.x == -1 && ij2.y == -1) return F2{-1, -1};
    if (ij2.x != -2 && ij2.y != -2) {
        int j0 = wrap_col(j - offhor * gap + GM, GM);
        int i0 = (i - offver * gap);
        F2 ij0 = g.at(i0, j0);
        if (ij0.x < 0) return F2{-1, -1};
        int jprev = wrap_col(j - 3 * offhor * gap + GM, GM);
        int jnext = wrap_col(j + 3 * offhor * gap + GM, GM);
        int iprev = i - offver * 3 * gap;
        int inext = i + offver * 3 * gap;
        if (offver != 0) {
            if (i2 == 0) {
                jnext = wrap_col(j0 + GM / 2, GM);
                inext = i0;
            } else if (i0 == GN - 1) {
                jprev = wrap_col(j0 + GM / 2, GM);
                iprev = i2;
            } else if (i2 == GN - 1) {
                inext = i0;
                jnext = wrap_col(j0 + GM / 2, GM);
            }
        }
        F2 ijprev = g.at(iprev, jprev);
        F2 ijnext = g.at(inext, jnext);
        if (ijprev.x > -2 && ijnext.x > -2) {
            F2 pt[4] = {ijprev, ij0, ij2, ijnext};
            if (pt[0].x != -1 && pt[3].x != -1) {
                pi_check_tot(pt, 0.2f, 4);
                return hermite(0.5f, pt[0], pt[1], pt[2], pt[3]);
            }
        }
        F2 pt[2] = {ij2, ij0};
        pi_check_tot(pt, 0.2f, 2);
        return F2{.5f * (pt[0].x + pt[1].x), .5f * (pt[0].y + pt[1].y)};
    }
    if (COUNT > 0) return F2{-1.f, -1.f};
    int j0 = wrap_col(j + gap, GM);
    int j1 = wrap_col(j - gap + GM, GM);
    if (i - gap < 0) return F2{-1, -1};
    const F2 c0 = g.at(i + gap, j0), c1 = g.at(i - gap, j0), c2 = g.at(i - gap, j1), c3 = g.at(i + gap, j1);
    if (c0.x == -1 || c0.x == -2 || c1.x == -1 || c1.x == -2 || c2.x == -1 || c2.x == -2 || c3.x == -1 || c3.x == -2)
        return F2{-1, -1};
    return interpolate_hermite_l1(g, i - gap, j1, 2 * gap, c0, c1, c2, c3);
}

// kernel.cuh:891-938 for recursion depth COUNT.  The eight outer points load
// together; the missing ones are then looked for.
template <int COUNT>
__device__ __forceinline__ F2 interpolate_hermite(const GridV& g, int i, int j, int gap, float percDown,
                                                  float percRight, F2* c) {
    const int GM = g.GM, GN = g.GN;
    int k = i + gap;
    int l = wrap_col(j + gap, GM);
    int imin1 = i - gap;
    int kplus1 = k + gap;
    int jmin1 = wrap_col(j - gap + GM, GM);
    int lplus1 = wrap_col(l + gap, GM);
    int jx = j, jy = j, lx = l, ly = l;
    if (i == 0) {
        jx = wrap_col(j + GM / 2, GM);
        lx = wrap_col(jx + gap, GM);
        imin1 = k;
    } else if (k == GN - 1) {
        jy = wrap_col(j + GM / 2, GM);
        ly = wrap_col(jy + gap, GM);
        kplus1 = i;
    }
    const int pi[8] = {i, i, k, k, imin1, imin1, kplus1, kplus1};
    const int pj[8] = {jmin1, lplus1, jmin1, lplus1, jx, lx, jy, ly};
    bool missing = false;
#pragma unroll
    for (int q = 0; q < 8; q++) c[4 + q] = g.at(pi[q], pj[q]);
#pragma unroll
    for (int q = 0; q < 8; q++) missing = missing || (c[4 + q].x == -2 && c[4 + q].y == -2);
    if (missing) {
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (c[4 + q].x == -2 && c[4 + q].y == -2)
                c[4 + q] = find_missing<COUNT>(g, pi[q], pj[q], q < 4 ? 0 : q < 6 ? -1 : 1,
                                               q >= 4 ? 0 : q % 2 ? 1 : -1, gap);
    }
    for (int q = 4; q < 12; q++)
        if (c[q].x == -1) return interpolate_linear(percDown, percRight, c);
    pi_check_tot(c, 0.2f, 12);
    F2 up = hermite(percRight, c[4], c[0], c[1], c[5]);
    F2 down = hermite(percRight, c[6], c[2], c[3], c[7]);
    F2 upup = F2{c[8].x + (c[9].x - c[8].x) * percRight, c[8].y + (c[9].y - c[8].y) * percRight};
    F2 downdown = F2{c[10].x + (c[11].x - c[10].x) * percRight, c[10].y + (c[11].y - c[10].y) * percRight};
    return hermite(percDown, upup, up, down, downdown);
}

__device__ __attribute__((noinline)) F2 interpolate_hermite_l1(GridV g, int i, int j, int gap, F2 c0, F2 c1, F2 c2,
                                                               F2 c3) {
    F2 c[12] = {c0, c1, c2, c3};
    return interpolate_hermite<1>(g, i, j, gap, .5f, .5f, c);
}

// MakeImageKernel.cu:328-351 with findBlock (kernel.cuh:736-752) and
// interpolateSpline (kernel.cuh:940-968).
__device__ F2 interpolate_pix(const GridV& g, float theta, float phi, int gridlvl, int& gapsave) {
    const int GM = g.GM;
    int half = (phi < BT_FPI) ? 0 : 1;
    int a = 0;
    int b = half * GM / 2;
    int gap = GM / 2;
    for (int s = 0; s < gridlvl + 1; s++) {
        int ngap = gap / 2;
        int k = a + ngap;
        int l = b + ngap;
        if (gap <= 1 || g.at(k, l).x == -2.f) break;
        // BT_FPI2 * k / (1.f * GM); for the usual power-of-two GM the division
        // is an exact scaling (two divisions were a third of a level's work)
        float thHalf = BT_FPI2 * k, phHalf = BT_FPI2 * l;
        if (g.inv != 0.f) {
            thHalf *= g.inv;
            phHalf *= g.inv;
        } else {
            thHalf /= 1.f * GM;
            phHalf /= 1.f * GM;
        }
        if (thHalf <= theta) a = k;
        if (phHalf <= phi) b = l;
        gap = ngap;
    }
    gapsave = gap;
    int k = a + gap;
    int l = b + gap;
    float factor = BT_FPI2 / (1.f * GM);
    float thetaUp = factor * a, phiLeft = factor * b, thetaDown = factor * k, phiRight = factor * l;
    l = wrap_col(l, GM);
    F2 c[12];
    c[0] = g.at(a, b);
    c[1] = g.at(a, l);
    c[2] = g.at(k, b);
    c[3] = g.at(k, l);
    F2 r;
    bool done = false;
    if (thetaUp == theta) {
        if (phiLeft == phi) {
            r = c[0];
            done = true;
        } else if (phiRight == phi) {
            r = c[1];
            done = true;
        } else if (a == 0.f) {
            r = c[0];
            done = true;
        }
    } else if (thetaDown == theta) {
        if (phiLeft == phi) {
            r = c[2];
            done = true;
        } else if (phiRight == phi) {
            r = c[3];
            done = true;
        }
    }
    if (!done) {
        bool captured = false;
        for (int q = 0; q < 4; q++)
            if (c[q].x == -1 && c[q].y == -1) captured = true;
        if (captured) {
            r = F2{-1.f, -1.f};
        } else {
            float percDown = (theta - thetaUp) / (thetaDown - thetaUp);
            float percRight = (phi - phiLeft) / (phiRight - phiLeft);
            r = interpolate_hermite<0>(g, a, b, gap, percDown, percRight, c);
        }
    }
    if (!(r.x == -1 && r.y == -1)) wrap_to_pi(r.x, r.y);
    return r;
}

// ------------------------------------------------------------------ kernels

__global__ __launch_bounds__(256) void pix_interp(GridV g, int gridlvl, const float* view, int W, int H,
                                                  float hor, float ver, float* thphi, int* gap) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i > H || j > W) return;
    size_t c = (size_t)i * (W + 1) + j;
    float theta = view[2 * c] + ver;
    float phi = fmod_2pi(view[2 * c + 1] + hor + BT_FPI2);
    int gs = 0;
    F2 r = interpolate_pix(g, theta, phi, gridlvl, gs);
    thphi[2 * c] = r.x;
    thphi[2 * c + 1] = r.y;
    gap[c] = gs;
}

// ---- multi-grid blending (G > 1): a frame between the poses of two grids
// A and B at fraction alpha (MakeImageKernel.cu:386-456,466-510).
//
// border (float2): [0] = (min, max) of pi/GN * i over the points captured in
// either grid, [1] the same of pi/GN * j (findBhCenter), both starting at
// (100, 0) (MakeImageKernel.cu:1308-1310); then for direction s, [2+2s] the
// shadow border of A and [3+2s] that of B (findBhBorders), box-smoothed
// four times (smoothBorder).  GN is the rows of the whole-sky grid.

// min i, max i, min j, max j of the captured points (ints: pi/GN * i is
// non-decreasing in i, so its extremes are those of i)
__global__ void bh_extent_init(int* ext) {
    if (threadIdx.x == 0) {
        ext[0] = 0x7fffffff;
        ext[1] = -1;
        ext[2] = 0x7fffffff;
        ext[3] = -1;
    }
}

__global__ __launch_bounds__(256) void bh_extent(GridV a, GridV b, int* ext) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = blockIdx.y * blockDim.y + threadIdx.y;
    const bool cap = i < a.GN && j < a.GM && (a.at(i, j).x == -1.f || b.at(i, j).x == -1.f);
    int v[4] = {cap ? i : 0x7fffffff, cap ? i : -1, cap ? j : 0x7fffffff, cap ? j : -1};
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        v[0] = min(v[0], __shfl_xor(v[0], off));
        v[1] = max(v[1], __shfl_xor(v[1], off));
        v[2] = min(v[2], __shfl_xor(v[2], off));
        v[3] = max(v[3], __shfl_xor(v[3], off));
    }
    if ((threadIdx.y * blockDim.x + threadIdx.x) % 64 == 0 && v[1] >= 0) {
        atomicMin(&ext[0], v[0]);
        atomicMax(&ext[1], v[1]);
        atomicMin(&ext[2], v[2]);
        atomicMax(&ext[3], v[3]);
    }
}

// findBhCenter's result from the extents, then findBhBorders: from the
// centre, step one grid unit at a time along direction s until a captured
// point is followed by a visible one.  The reference walks without a bound
// (and reads outside its grid when the walk leaves it); here the walk stops
// at the grid's edge.
__global__ __launch_bounds__(256) void bh_borders(GridV a, GridV b, const int* ext, float2* border) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * kAngleNum) return;
    const float gridsize = BT_FPI / (1.f * a.GN);
    float2 b0 = make_float2(100.f, 0.f), b1 = make_float2(100.f, 0.f);
    if (ext[1] >= 0) {
        b0 = make_float2(fminf(100.f, gridsize * (float)ext[0]), fmaxf(0.f, gridsize * (float)ext[1]));
        b1 = make_float2(fminf(100.f, gridsize * (float)ext[2]), fmaxf(0.f, gridsize * (float)ext[3]));
    }
    if (i == 0) {
        border[0] = b0;
        border[1] = b1;
    }
    const int ii = i / 2;
    const float angle = BT_FPI2 / (1.f * kAngleNum) * 1.f * ii;
    const float thetaChange = -f_sin(angle);
    const float phiChange = f_cos(angle);
    float ptx = .5f * b0.x + .5f * b0.y, pty = .5f * b1.x + .5f * b1.y;
    ptx = ptx / BT_FPI2 * (float)a.GM;
    pty = pty / BT_FPI2 * (float)a.GM;
    const GridV& g = (i % 2) ? b : a;
    float gA = -2.f, gB = -2.f;
    while (!(gA > 0 && gB == -1.f)) {
        gB = gA;
        ptx += thetaChange;
        pty += phiChange;
        const int gx = cvt_i32(ptx), gy = cvt_i32(pty);
        if (gx < 0 || gx >= g.GN || gy < 0 || gy >= g.GM) break;
        gA = g.at(gx, gy).x;
    }
    border[2 + i] = make_float2((ptx - thetaChange) * BT_FPI2 / (1.f * a.GM), (pty - phiChange) * BT_FPI2 / (1.f * a.GM));
}

// smoothBorder (MakeImageKernel.cu:444-456): mean of each border point and
// its two neighbours of the same grid
__global__ __launch_bounds__(256) void smooth_border(const float2* src, float2* dst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * kAngleNum) return;
    if (i == 0) {
        dst[0] = src[0];
        dst[1] = src[1];
    }
    const int prev = (i - 2 + 2 * kAngleNum) % (2 * kAngleNum);
    const int next = (i + 2) % (2 * kAngleNum);
    dst[i + 2] = make_float2(1.f / 3.f * (src[prev + 2].x + src[i + 2].x + src[next + 2].x),
                             1.f / 3.f * (src[prev + 2].y + src[i + 2].y + src[next + 2].y));
}

// pixInterpolation with Gr > 1 (MakeImageKernel.cu:466-510).  Inside the
// stretch circle around the shadow the two grids are sampled at positions
// warped so that their shadow borders meet the blended border.  The
// reference's direction slot can reach angleNum when the angle rounds to
// 2 pi (one entry past its border array); here it is clamped.
__global__ __launch_bounds__(256) void pix_interp_blend(GridV ga, GridV gb, int gridlvl, const float2* border,
                                                        float alpha, const float* view, int W, int H, float hor,
                                                        float ver, float* thphi, int* gap) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i > H || j > W) return;
    size_t c = (size_t)i * (W + 1) + j;
    float theta = view[2 * c] + ver;
    float phi = fmod_2pi(view[2 * c + 1] + hor + BT_FPI2);
    const float2 b0 = border[0], b1 = border[1];
    const float cx = .5f * b0.x + .5f * b0.y, cy = .5f * b1.x + .5f * b1.y;
    const float stretchRad = fmaxf(b0.y - b0.x, b1.x - b1.y) * 0.75f;
    const float centerdist = (theta - cx) * (theta - cx) + (phi - cy) * (phi - cy);
    int gs = 0;
    F2 A, B;
    if (centerdist < stretchRad * stretchRad) {
        float angle = f_atan2(cx - theta, phi - cy);
        angle = fmodf(angle + BT_FPI2, BT_FPI2);
        int slot = cvt_i32(angle / BT_FPI2 * (float)kAngleNum);
        slot = slot < 0 ? 0 : (slot >= kAngleNum ? kAngleNum - 1 : slot);
        const float2 bA = border[2 * slot + 2], bB = border[2 * slot + 3];
        const float nx = (1.f - alpha) * bA.x + alpha * bB.x;
        const float ny = (1.f - alpha) * bA.y + alpha * bB.y;
        if (centerdist <= (nx - cx) * (nx - cx) + (ny - cy) * (ny - cy)) {
            // inside the blended shadow; the reference leaves gap unwritten
            // here, and only shadow pixels touch this corner
            thphi[2 * c] = -1.f;
            thphi[2 * c + 1] = -1.f;
            gap[c] = 0;
            return;
        }
        const float tStoB = (cx - stretchRad * f_sin(angle) - nx);
        const float pStoB = (cy + stretchRad * f_cos(angle) - ny);
        // 1E-5 is a double in the reference: the comparison is in double
        const float thetaPerc = (double)fabsf(tStoB) < 1E-5 ? 0.f : 1.f - (theta - nx) / tStoB;
        const float phiPerc = (double)fabsf(pStoB) < 1E-5 ? 0.f : 1.f - (phi - ny) / pStoB;
        const float thetaA = theta - thetaPerc * (nx - bA.x);
        const float phiA = phi - phiPerc * (ny - bA.y);
        const float thetaB = theta - thetaPerc * (nx - bB.x);
        const float phiB = phi - phiPerc * (ny - bB.y);
        A = interpolate_pix(ga, thetaA, phiA, gridlvl, gs);
        B = interpolate_pix(gb, thetaB, phiB, gridlvl, gs);
    } else {
        A = interpolate_pix(ga, theta, phi, gridlvl, gs);
        B = interpolate_pix(gb, theta, phi, gridlvl, gs);
    }
    F2 r;
    if (A.x == -1.f || B.x == -1.f) {
        r = F2{-1.f, -1.f};
    } else {
        if (A.y < .2f * BT_FPI2 && B.y > .8f * BT_FPI2) A.y += BT_FPI2;
        if (B.y < .2f * BT_FPI2 && A.y > .8f * BT_FPI2) B.y += BT_FPI2;
        r = F2{(1.f - alpha) * A.x + alpha * B.x, fmodf((1.f - alpha) * A.y + alpha * B.y, BT_FPI2)};
    }
    thphi[2 * c] = r.x;
    thphi[2 * c + 1] = r.y;
    gap[c] = gs;   // the second lookup's, as the reference's writes land in that order
}

// kernel.cuh:652-672; false when a corner is negative (shadow).
__device__ __forceinline__ bool corners(const float* thphi, int W, int ind, float* t, float* p,
                                        bool& picheck, float offset) {
    const int M1 = W + 1;
    const float2* tp = reinterpret_cast<const float2*>(thphi);
    float2 c0 = tp[ind + M1], c1 = tp[ind], c2 = tp[ind + 1], c3 = tp[ind + M1 + 1];
    t[0] = c0.x; t[1] = c1.x; t[2] = c2.x; t[3] = c3.x;
    p[0] = c0.y; p[1] = c1.y; p[2] = c2.y; p[3] = c3.y;
    for (int q = 0; q < 4; q++) {
        if (p[q] < 0 || t[q] < 0) return false;
        p[q] = fmod_2pi(p[q] + offset);
    }
    picheck = pi_check(p, .2f);
    return true;
}

// The solid angle of a shadow pixel while the smoothing runs (a real one lies
// within +-4 pi or is no number): the filters then read one array.
constexpr float kShadowArea = -3.0e38f;

// Unit vectors of the (16 + 1) x (16 + 1) corners of a 16 x 16 tile of
// quads, in LDS: four quads share a corner, and its FP64 sines and cosines
// are most of the work on a solid angle.
struct TileVec {
    float x[17 * 17], y[17 * 17], z[17 * 17];
    __device__ __forceinline__ void set(int c, float t, float p) {
        const float sint = f_sin(t);
        x[c] = sint * f_cos(p);
        y[c] = sint * f_sin(p);
        z[c] = f_cos(t);
    }
    __device__ __forceinline__ void get(const int* c, float* xi, float* yi, float* zi, int n) const {
        for (int q = 0; q < n; q++) {
            xi[q] = x[c[q]];
            yi[q] = y[c[q]];
            zi[q] = z[c[q]];
        }
    }
};

// Shadow flag and celestial solid angle (findBlackPixels + findArea).  The
// pixel across phi = 2 pi, whose corners pi_check moves, makes its own
// vectors.  Also clears the counters of the star and sky queues of the frame.
__global__ __launch_bounds__(256) void bh_area(const float* thphi, int W, int H, uint8_t* bh, float* area,
                                               unsigned* ctr, int nctr) {
    __shared__ TileVec V;
    const int tid = threadIdx.y * 16 + threadIdx.x;
    if (blockIdx.x == 0 && blockIdx.y == 0)
        for (int k = tid; k < nctr; k += 256) ctr[k] = 0u;
    const float2* tp = reinterpret_cast<const float2*>(thphi);
    for (int c = tid; c < 17 * 17; c += 256) {
        const int ci = blockIdx.y * 16 + c / 17, cj = blockIdx.x * 16 + c % 17;
        if (ci > H || cj > W) continue;
        const float2 v = tp[(size_t)ci * (W + 1) + cj];
        if (!(v.x < 0 || v.y < 0)) V.set(c, v.x, fmod_2pi(v.y + 0.0f));
    }
    __syncthreads();
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= H || j >= W) return;
    float t[4], p[4];
    bool pc = false;
    bool ok = corners(thphi, W, i * (W + 1) + j, t, p, pc, 0.0f);
    size_t ij = (size_t)i * W + j;
    bh[ij] = ok ? 0 : 1;
    float a = kShadowArea;
    if (ok && pc) {
        a = quad_area_cold(t[0], t[1], t[2], t[3], p[0], p[1], p[2], p[3]);
    } else if (ok) {
        const int o = threadIdx.y * 17 + threadIdx.x;
        const int c0[3] = {o + 17, o, o + 1}, c1[3] = {o + 17, o + 1, o + 18};
        float x[3], y[3], z[3];
        V.get(c0, x, y, z, 3);
        a = area3_of(x, y, z);
        V.get(c1, x, y, z, 3);
        a = a + area3_of(x, y, z);
    }
    area[ij] = a;
}

__device__ __forceinline__ int filter_size(const int* gap, int W, int i, int j) {
    const int M1 = W + 1;
    int fs = gap[i * M1 + j];
    fs = max(fs, gap[i * M1 + M1 + j]);
    fs = max(fs, gap[i * M1 + j + 1]);
    fs = max(fs, gap[i * M1 + M1 + j + 1]);
    return fs / 2;
}

// MakeImageKernel.cu:570-591.  Four taps' loads are in flight together; the
// sum stays in tap order (a shadow tap adds a zero).
__global__ __launch_bounds__(256) void smooth_h(const float* area, const int* gap, int W, int H, float* area_s) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= H || j >= W) return;
    size_t ij = (size_t)i * W + j;
    const float own = area[ij];
    if (own == kShadowArea) {
        area_s[ij] = kShadowArea;
        return;
    }
    const int fs = filter_size(gap, W, i, j);
    const float* row = area + (size_t)i * W;
    float sum = 0.f;
    int count = 0;
    int jj = j - fs;
    while (jj < 0) jj += W;   // at most one step unless the filter is wider than the frame
    for (int h = 0; h <= 2 * fs; h += 4) {
        float x[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            x[u] = h + u <= 2 * fs ? row[jj] : kShadowArea;
            jj = jj + 1 >= W ? 0 : jj + 1;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const bool lit = x[u] != kShadowArea;
            sum += lit ? x[u] : 0.f;
            count += lit;
        }
    }
    area_s[ij] = sum / (1.f * count);
}

// MakeImageKernel.cu:593-616
__global__ __launch_bounds__(256) void smooth_v(const float* area_s, const int* gap, int W, int H, float* area) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= H || j >= W) return;
    size_t ij = (size_t)i * W + j;
    const float own = area_s[ij];
    if (own == kShadowArea) {
        area[ij] = 0.f;
        return;
    }
    const int fs = filter_size(gap, W, i, j);
    const int minv = max(0, i - fs);
    const int maxv = min(H - 1, i + fs);
    float sum = 0.f;
    int count = 0;
    for (int h = minv; h <= maxv; h += 4) {
        float x[4];
#pragma unroll
        for (int u = 0; u < 4; u++) x[u] = h + u <= maxv ? area_s[(size_t)(h + u) * W + j] : kShadowArea;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const bool lit = x[u] != kShadowArea;
            sum += lit ? x[u] : 0.f;
            count += lit;
        }
    }
    area[ij] = sum / (1.f * count);
}

// kernel.cuh:674-692
__device__ void lensing_redshift(const float* t, const float* p, int W, int ind, const Cam7& cam,
                                 const float* view, float& frac, float& redshft, float solidAngle) {
    const int M1 = W + 1;
    if (solidAngle == 0.f)
        solidAngle = quad_area_cold(t[0], t[1], t[2], t[3], p[0], p[1], p[2], p[3]);
    const float2* v = reinterpret_cast<const float2*>(view);
    float2 v0 = v[ind], v1 = v[ind + 1], v2 = v[ind + M1 + 1], v3 = v[ind + M1];
    float ver4[4] = {v0.x, v1.x, v2.x, v3.x};
    float hor4[4] = {v0.y, v1.y, v2.y, v3.y};
    // area4_of these corners, made once per view (view_pixel_areas)
    const int pi = ind / M1, pj = ind - pi * M1;
    const float pixArea = cam.pix_area[(size_t)pi * W + pj];
    frac = pixArea / solidAngle;
    float thetaCam = (ver4[0] + ver4[1] + ver4[2] + ver4[3]) * .25f;
    float phiCam = (hor4[0] + hor4[1] + hor4[2] + hor4[3]) * .25f;
    redshft = redshift(thetaCam, phiCam, cam.v);
}

// The camera-sky solid angle of every pixel's view quad (the pixArea of
// kernel.cuh:679-680): it depends on the view alone, so a view makes it once.
__global__ __launch_bounds__(256) void view_pixel_areas(const float* view, int W, int H, float* out) {
    __shared__ TileVec V;
    const int M1 = W + 1;
    const float2* v = reinterpret_cast<const float2*>(view);
    for (int c = threadIdx.y * 16 + threadIdx.x; c < 17 * 17; c += 256) {
        const int ci = blockIdx.y * 16 + c / 17, cj = blockIdx.x * 16 + c % 17;
        if (ci > H || cj > W) continue;
        const float2 d = v[(size_t)ci * M1 + cj];
        V.set(c, d.x, d.y);
    }
    __syncthreads();
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= H || j >= W) return;
    const int o = threadIdx.y * 17 + threadIdx.x;
    const int c4[4] = {o, o + 1, o + 18, o + 17};
    float x[4], y[4], z[4];
    V.get(c4, x, y, z, 4);
    out[(size_t)i * W + j] = area4_of(x, y, z);
}

// ---- star pass ---------------------------------------------------------
// distortStarMap (MakeImageKernel.cu:206-326).
//
// Candidates.  The reference tests every star of the star-tree nodes that
// overlap a pixel's quad bounding box (searchTree, MakeImageKernel.cu:27-96):
// ~390 stars per level-8 leaf for a quad of ~1e-3 rad.  Any superset of the
// stars inside the quad yields the same inside-star set, so pixels read
// candidates from a 256 x 512 (theta, phi) binning of the stars instead:
// one contiguous range per bin row, ~1 star per bin.  The exception is a
// quad that crosses phi = 2 pi (picheck): there the reference retests
// candidates with phi < 0.4 pi shifted by 2 pi, so which stars are
// candidates matters, and those pixels walk the reference's tree.
//
// Work split.  Near the shadow a pixel can project onto a large part of the
// sky with tens of thousands of candidates; one lane would serialise them and
// stall its wavefront.  star_scan finds the pixels with at most kLightStars
// candidates and a star inside (5% of the pixels of a lensed 1080p frame;
// star_few traces them, one lane each), and queues those with more (6%),
// whose candidates star_map_chunk splits over wavefronts, the taps reduced in
// a fixed order.
//
// Per tap the reference evaluates 100 * 10^(-0.4 (m - 2.5 log10 x)) with
// x = frac * gaussian(d) and converts HSP -> RGB at brightness P * that.
// For finite x > 0 this equals 100 * x * 10^(-0.4 m), and HSP -> RGB is
// linear in P, so the colour is converted once per star and each tap is a
// few multiplies; non-finite or non-positive x (which yield 0 or NaN in the
// reference) take the reference's own expression.  The star light agrees
// with the reference arithmetic to a few ulps up to summation order; frames
// to within 1/255.
constexpr int kLightStars = 16;

// Appends `value` to list for every lane with `take` set: one atomic per
// wavefront.  Every active lane of the wave must call it.
__device__ __forceinline__ void wave_append(uint32_t* list, unsigned* count, bool take, uint32_t value) {
    const unsigned lane = __lane_id();
    unsigned long long m = __ballot(take);
    if (!m) return;
    const int leader = __ffsll((long long)m) - 1;
    unsigned base = 0;
    if (lane == (unsigned)leader) base = atomicAdd(count, (unsigned)__popcll(m));
    base = __shfl(base, leader);
    if (take) list[base + (unsigned)__popcll(m & ((1ull << lane) - 1))] = value;
}

struct StarPix {
    const float* colours;   // star_colours table (6 floats per blackbody index)
    float t[4], p[4];
    float mn[2], mx[2];
    int sgn;
    bool picheck;
    bool odd;   // lensing out of the range where every tap takes the fast form
    float frac, redshft, red;
};

// Per blackbody index: rgb_to_hsp of the table colour (H, S, P) and
// hsp_to_rgb of that at the same P (R, G, B) -- what every star of that
// colour would compute (kernel.cuh:451-468), once.
__global__ void star_colours(float* out) {
    int index = blockIdx.x * blockDim.x + threadIdx.x;
    if (index > 390) return;
    float hh, ss, pp, r1, g1, b1;
    rgb_to_hsp((float)kTempRGB[3 * index] / 255.f, (float)kTempRGB[3 * index + 1] / 255.f,
               (float)kTempRGB[3 * index + 2] / 255.f, hh, ss, pp);
    hsp_to_rgb(hh, ss, pp, r1, g1, b1);
    float* o = out + 6 * index;
    o[0] = hh;
    o[1] = ss;
    o[2] = pp;
    o[3] = r1;
    o[4] = g1;
    o[5] = b1;
}

// Corners, bounding box and orientation of pixel (i, j) (no lensing).
__device__ void star_pixel_geom(const float* thphi, int W, int i, int j, float offset, const Cam7& cam,
                                StarPix& P) {
    P.colours = cam.colours;
    const int ind = i * (W + 1) + j;
    P.picheck = false;
    corners(thphi, W, ind, P.t, P.p, P.picheck, offset);
    const float* t = P.t;
    const float* p = P.p;
    P.mx[0] = fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]));
    P.mx[1] = fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]));
    P.mn[0] = fminf(fminf(t[0], t[1]), fminf(t[2], t[3]));
    P.mn[1] = fminf(fminf(p[0], p[1]), fminf(p[2], p[3]));
    float orient = (t[1] - t[0]) * (p[1] + p[0]) + (t[2] - t[1]) * (p[2] + p[1]) + (t[3] - t[2]) * (p[3] + p[2]) +
                   (t[0] - t[3]) * (p[0] + p[3]);
    P.sgn = orient < 0 ? -1 : 1;
}

// Lensing factor and redshift of the pixel whose corners P holds.
__device__ __forceinline__ void star_lens(int W, size_t ij, int ind, int lr, const float* area, const float* view,
                                          const Cam7& cam, StarPix& P) {
    P.redshft = 1.f;
    P.frac = 1.f;
    if (lr) lensing_redshift(P.t, P.p, W, ind, cam, view, P.frac, P.redshft, area[ij]);
    P.red = 4.f * log10f(P.redshft);   // device library FP32 (a few ulps)
}

__device__ bool star_pixel(const float* thphi, const uint8_t* bh, int W, int i, int j, float offset, int lr,
                           const float* area, const float* view, const Cam7& cam, StarPix& P) {
    const size_t ij = (size_t)i * W + j;
    if (bh[ij] != 0) return false;
    star_pixel_geom(thphi, W, i, j, offset, cam, P);
    star_lens(W, ij, i * (W + 1) + j, lr, area, view, cam, P);
    return true;
}

__device__ __forceinline__ void node_range(const int32_t* tree, int node, int& b, int& e) {
    b = (node != 0 && ((node + 1) & node) != 0) ? tree[node - 1] : 0;
    e = tree[node];
}

// searchTree (MakeImageKernel.cu:27-96) with picheck = 0: visit(node) is
// called for every listed node in the reference's list order.  The node's
// rectangle is held in scalars (0: theta, 1: phi), not in arrays indexed by
// the level's axis, which would live in scratch memory.
// The walk ends early once done() holds.
template <class F, class D>
__device__ void search_tree_until(const int32_t* tree, int treeLevel, const float* mn, const float* mx, F&& visit,
                                  D&& done) {
    float start0 = 0.f, start1 = 0.f, size0 = BT_FPI, size1 = BT_FPI2;
    int node = 0;
    unsigned bitMask = 1u << treeLevel;
    int level = 0;
    int lvl = 0;
    while (bitMask != 0) {
        bitMask &= ~(1u << (treeLevel - level));
        for (lvl = level + 1; lvl <= treeLevel; lvl++) {
            int star_n = tree[node];
            if (node != 0 && ((node + 1) & node) != 0) star_n -= tree[node - 1];
            const bool ph = (lvl & 1) != 0;
            const float full0 = size0, full1 = size1;
            if (ph) size1 = size1 * .5f;
            else size0 = size0 * .5f;
            if (star_n == 0) {
                node = node * 2 + 1;
                break;
            }
            float check = ph ? start1 + size1 : start0 + size0;
            bool lu = (ph ? mn[1] : mn[0]) < check;
            bool rd = (ph ? mx[1] : mx[0]) >= check;
            bool list = lvl == treeLevel;
            if (!list && rd && lu) {   // the quad covers most of the node
                float x_overlap = fmaxf(0.f, fminf(mx[0], start0 + full0) - fmaxf(mn[0], start0));
                float y_overlap = fmaxf(0.f, fminf(mx[1], start1 + full1) - fmaxf(mn[1], start1));
                float overlapArea = x_overlap * y_overlap;
                list = overlapArea / (full0 * full1) > 0.8f;
            }
            if (list) {
                if (rd) visit(node * 2 + 2);
                if (lu) visit(node * 2 + 1);
                if (done()) return;
                node = node * 2 + 1;
                break;
            } else {
                node = node * 2 + 1;
                if (rd) bitMask |= 1u << (treeLevel - lvl);
                if (!lu) break;
            }
        }
        level = treeLevel - (__ffs((int)bitMask)) + 1;
        if (level >= 0) {
            int diff = lvl - level;
            for (int q = 0; q < diff; q++) {
                if ((lvl - q) & 1) {
                    if (!(node & 1)) start1 -= size1;
                    size1 = size1 * 2.f;
                } else {
                    if (!(node & 1)) start0 -= size0;
                    size0 = size0 * 2.f;
                }
                node = (node - 1) / 2;
            }
            node++;
            if (level & 1) start1 += size1;
            else start0 += size0;
        }
    }
}

template <class F>
__device__ void search_tree(const int32_t* tree, int treeLevel, const float* mn, const float* mx, F&& visit) {
    search_tree_until(tree, treeLevel, mn, mx, visit, [] { return false; });
}

__device__ __forceinline__ int bin_of(float v, float d, int n) { return min(max(cvt_i32(v / d), 0), n - 1); }

// The phi bins [q0, q1] of bin row r (theta in [r, r + 1] * kBinDT) that can
// hold a star passing star_in_polygon, within the pixel's bounding-box bins
// [p0, p1]; q0 > q1 when none can.  Each edge test of star_in_polygon,
// A (sp - p_b) - B (st - t_b) > 0 with A = sgn (t_a - t_b) and
// B = sgn (p_a - p_b), bounds phi by a line in theta whose extremes over the
// row are at its two ends; the four bounds are intersected.  Conservative:
// the row is widened by 1e-3 of a bin in theta, the span by one bin on each
// side (the rounding of the FP32 edge tests is far below a bin), and an edge
// that is steep in this frame (|B| > 1000 |A|, where that rounding divided by
// |A| could reach a bin) bounds nothing.  On a strongly lensed pixel (a thin
// arc of the Einstein ring) this tests a small fraction of its bounding
// box's stars.
struct EdgeLines {
    float g[4];      // dphi/dtheta of edge k's line
    unsigned side;   // bit k: it bounds phi from below; bit 4 + k: from above
    __device__ __forceinline__ void set(const StarPix& P) {
        const float sg = (float)P.sgn;
        side = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int kb = (k + 1) & 3;
            const float A = sg * (P.t[k] - P.t[kb]);
            const float B = sg * (P.p[k] - P.p[kb]);
            g[k] = B / A;
            if (fabsf(B) <= 1000.f * fabsf(A)) side |= A > 0.f ? 1u << k : 16u << k;   // not A == 0, NaN
        }
    }
};

__device__ __forceinline__ void row_span(const float* t, const float* p, float mn1, float mx1, const EdgeLines& L,
                                         int r, int p0, int p1, int& q0, int& q1) {
    const float ta = ((float)r - 1e-3f) * kBinDT, tb = ((float)r + 1.001f) * kBinDT;
    float lo = mn1, hi = mx1;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int kb = (k + 1) & 3;
        const float la = p[kb] + L.g[k] * (ta - t[kb]);
        const float lb = p[kb] + L.g[k] * (tb - t[kb]);
        if (L.side & (1u << k)) lo = fmaxf(lo, fminf(la, lb));
        if (L.side & (16u << k)) hi = fminf(hi, fmaxf(la, lb));
    }
    if (!(lo <= hi)) {
        q0 = 1;
        q1 = 0;
        return;
    }
    q0 = max(p0, bin_of(lo, kBinDP, kBinP) - 1);
    q1 = min(p1, bin_of(hi, kBinDP, kBinP) + 1);
}

// The candidates [b, e) of bin row r (none beyond row r1).
__device__ __forceinline__ void row_bounds(const StarPix& P, const EdgeLines& L, const SceneK& s, int r, int r1, int p0,
                                           int p1, int& b, int& e) {
    b = e = 0;
    if (r > r1) return;
    int q0, q1;
    row_span(P.t, P.p, P.mn[1], P.mx[1], L, r, p0, p1, q0, q1);
    if (q0 <= q1) {
        b = s.bin_start[r * kBinP + q0];
        e = s.bin_start[r * kBinP + q1 + 1];
    }
}

// f(begin, end) for every candidate range of a pixel; ranges index
// ranges_pos/ranges_mag (tree order for picheck pixels, bin order otherwise).
template <class F>
__device__ void for_ranges(const StarPix& P, const SceneK& s, F&& f) {
    if (P.picheck) {
        search_tree(s.tree, s.tree_level, P.mn, P.mx, [&](int node) {
            int b, e;
            node_range(s.tree, node, b, e);
            f(b, e);
        });
    } else {
        const int r0 = bin_of(P.mn[0], kBinDT, kBinT), r1 = bin_of(P.mx[0], kBinDT, kBinT);
        const int p0 = bin_of(P.mn[1], kBinDP, kBinP), p1 = bin_of(P.mx[1], kBinDP, kBinP);
        EdgeLines L;
        L.set(P);
        // four rows' bounds load together
        for (int r = r0; r <= r1; r += 4) {
            int b[4], e[4];
#pragma unroll
            for (int k = 0; k < 4; k++) row_bounds(P, L, s, r + k, r1, p0, p1, b[k], e[k]);
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (b[k] < e[k]) f(b[k], e[k]);
        }
    }
}

// The inside test of one candidate star (MakeImageKernel.cu:285-292): st,
// sp receive its position (phi shifted by 2 pi for the retest of a quad
// across phi = 2 pi).
__device__ __forceinline__ bool star_test(const StarPix& P, const float* pos, int q, float& st, float& sp) {
    const float2 sp2 = reinterpret_cast<const float2*>(pos)[q];
    st = sp2.x;
    sp = sp2.y;
    bool in = star_in_polygon(P.t, P.p, st, sp, P.sgn);
    if (P.picheck && !in && sp < BT_FPI2 * .2f) {
        sp += BT_FPI2;
        in = star_in_polygon(P.t, P.p, st, sp, P.sgn);
    }
    return in;
}

// 10^x in FP32 to a few ulps: 2^(x log2 10), the product carried in two
// parts (log2 10 = L1 + L2, the rounding of x L1 recovered by an FMA), so
// that the exponent's rounding (large for large |x|) does not reach the
// result.
__device__ __forceinline__ float exp10_f32(float x) {
    constexpr float L1 = 3.32192802429199219f;     // log2(10) rounded to float
    constexpr float L2 = 7.05797954e-08f;          // log2(10) - L1
    const float hi = x * L1;
    const float lo = fmaf(x, L1, -hi) + x * L2;
    return exp2f(hi) * (1.f + lo * 0.693147180559945309f);
}

// Whether every tap of every star takes the fast form in this pixel: the
// tap weight x = frac * gaussian(d) lies in [0, 3.4e38] for frac in
// [1e-30, 1e30] (over the footprints of steps 1, 2 and 3 gaussian(d) falls
// from 1 to 8.8e-4, 3.3e-9 and 2.4e-17; an x that underflows to zero is no
// light in either form), and E = 10^(-0.4 (m + red)) stays finite for
// m >= -10, |red| <= 80.
__device__ __forceinline__ bool star_pixel_odd(const StarPix& P, const SceneK& s) {
    return !(s.mag_tame && P.frac >= 1e-30f && P.frac <= 1e30f && P.red >= -80.f && P.red <= 80.f);
}

// The reference's own expression for one tap (kernel.cuh:390,
// MakeImageKernel.cu:310-318).  Out of line: its FP64 log and pow inlined in
// every tap make the odd kernels larger than the instruction cache, and they
// then wait for their own code (the odd chunks of a 320x180 frame took 250 us).
struct Rgb {
    float r, g, b;
};
__device__ __attribute__((noinline)) Rgb star_tap_slow(float part, float x, float hh, float ss, float pp) {
    const float appMag = part - 2.5f * f_log10(x);
    const float brightness = 100 * f_exp10(-.4f * appMag);
    Rgb o;
    hsp_to_rgb(hh, ss, pp * brightness, o.r, o.g, o.b);
    return o;
}

// The light of one star inside the pixel (MakeImageKernel.cu:293-322).
// Per tap the reference evaluates 100 * 10^(-0.4 (part - 2.5 log10 x)) with
// x = frac * gaussian(d); for finite x > 0 and finite E = 10^(-0.4 part)
// that is 100 x E.  ODD = false (pixels where star_pixel_odd is false):
// every tap takes that fast form.  ODD = true: each tap checks, and takes
// the reference's own expression (kernel.cuh:390, MakeImageKernel.cu:310-318)
// where the fast form does not apply.
template <int STEP, bool ODD>
__device__ __forceinline__ void star_splat(const StarPix& P, const float* mag, int q, float st, float sp,
                                           float (&acc)[(2 * STEP + 1) * (2 * STEP + 1)][3]) {
    constexpr int FW = 2 * STEP + 1;
    interpolate_star(P.t[0], P.t[1], P.t[2], P.t[3], P.p[0], P.p[1], P.p[2], P.p[3], st, sp, P.sgn);
    const float2 mg = reinterpret_cast<const float2*>(mag)[q];
    const float part = mg.x + P.red;
    float temp = 46.f / P.redshft * ((1.f / ((0.92f * mg.y) + 1.7f)) + (1.f / ((0.92f * mg.y) + 0.62f))) - 10.f;
    // clamp to the table's last entry (the reference's 1170 reads past it)
    int index = max(0, min(cvt_i32(floorf(temp)), 390));
    // the blackbody colour's HSP and its RGB at unit brightness, per index
    const float* col = P.colours + 6 * index;
    const float r1 = col[3], g1 = col[4], b1 = col[5];
    const float E = ODD ? f_exp10(-.4f * part) : exp10_f32(-.4f * part);
    const float maxDistSq = (STEP + .5f) * (STEP + .5f);
    // A lensing factor that is no positive finite number makes every tap's x
    // the same infinity, zero or (log of a negative) NaN: one slow evaluation
    // serves them all.
    const bool flat = ODD && !(P.frac > 0.f && P.frac <= 3.4e38f);
    Rgb all{0.f, 0.f, 0.f};
    if (flat) all = star_tap_slow(part, P.frac, col[0], col[1], col[2]);
#pragma unroll
    for (int u = 0; u < FW; u++)
#pragma unroll
        for (int v = 0; v < FW; v++) {
            float dt = -STEP + u + .5f - st;
            float dp = -STEP + v + .5f - sp;
            float dist = dt * dt + dp * dp;
            if (dist > maxDistSq) continue;
            float x = P.frac * gaussian(dist);
            float rr, gg, bb;
            if (!ODD || (x > 0.f && x <= 3.4e38f && fabsf(E) <= 3.4e38f)) {
                float bright = 100.f * x * E;
                rr = r1 * bright;
                gg = g1 * bright;
                bb = b1 * bright;
            } else {
                const Rgb o = flat ? all : star_tap_slow(part, x, col[0], col[1], col[2]);
                rr = o.r;
                gg = o.g;
                bb = o.b;
            }
            rr *= 255.f;
            gg *= 255.f;
            bb *= 255.f;
            acc[FW * u + v][0] += rr * rr;
            acc[FW * u + v][1] += gg * gg;
            acc[FW * u + v][2] += bb * bb;
        }
}

// One candidate star of one pixel (the body of MakeImageKernel.cu:285-322).
template <int STEP, bool ODD>
__device__ __forceinline__ void star_accumulate(const StarPix& P, const float* pos, const float* mag, int q,
                                                float (&acc)[(2 * STEP + 1) * (2 * STEP + 1)][3]) {
    float st, sp;
    if (star_test(P, pos, q, st, sp)) star_splat<STEP, ODD>(P, mag, q, st, sp, acc);
}

// Pixels with more than kLightStars candidates are queued with their
// candidate count and cut into chunks of kChunk candidates, one wavefront
// per chunk; their chunk indices are taken by an atomic in star_assign
// (contiguous per pixel).  A pixel's chunk partials are summed in
// chunk order, so the result does not depend on which waves ran which
// chunks.  (Where a frame has more chunks than pixels, one lane adds up the
// pixels whose chunks found no room, candidate by candidate; which those are
// depends on the order of the atomics, and with it the last bits of their
// sums.)  Every queued star is then
// one of a few candidates of one lane, whatever the pixel it lands in: the
// long per-star chain (bisection, taps) of a pixel with tens of thousands of
// candidates is spread over many waves instead of serialised on a few lanes.
constexpr int kChunk = 256;

// A queued count with this bit set is a pixel whose candidates come from
// the star tree (a quad across phi = 2 pi).  star_wide walks the tree for
// such a pixel and stores its listed node ranges, so that every chunk of the
// pixel walks the stored ranges as a binned pixel walks its bin rows.
constexpr uint32_t kTreePixel = 0x80000000u;
// A queued count with this bit set is an odd pixel (star_pixel_odd): its
// chunks are traced by the ODD instance of star_map_chunk.
constexpr uint32_t kOddPixel = 0x40000000u;

__device__ __forceinline__ uint32_t queued_count(uint32_t v) { return v & ~(kTreePixel | kOddPixel); }
__device__ __forceinline__ uint32_t queued_chunks(uint32_t v) { return (queued_count(v) + kChunk - 1) / kChunk; }

// owner of a chunk index that star_map_chunk<false> passes over: taken by a
// pixel whose chunks did not all fit `cap` (one lane traces it), or by an odd
// pixel
constexpr uint32_t kNoOwner = 0xffffffffu;

struct StarQueue {
    uint32_t* pix;         // queued pixel indices
    uint32_t* cnt;         // their candidate counts (| kTreePixel | kOddPixel); 0: no chunk work
    uint32_t* nnode;       // tree pixels: listed node count
    uint32_t* rbase;       // tree pixels: first stored range
    int2* ranges;          // stored node ranges (begin, end) of tree pixels
    unsigned rcap;         // capacity of `ranges`
    uint32_t* cstart;      // first chunk of each queued pixel
    uint32_t* owner;       // queued pixel of each chunk (or kNoOwner)
    float* lens;           // per queued pixel: frac, redshift, 4 log10(redshift)
    uint32_t* wide;        // queue entries that star_wide counts: binned ones from the front, tree ones from the back
                           // (NP + 64 of them, in owner's memory)
    uint32_t* odd;         // pixels for star_map_odd
    uint32_t* oddc;        // chunks of odd pixels (in the smoothing's memory)
    unsigned* ctr;         // the counters below, each on a line of its own
    float* partial;        // per chunk: FW*FW*3 partial taps
    unsigned cap;          // chunk capacity of `partial`
    uint8_t* lit;          // per pixel: kDark, or who writes its taps this frame
};
// StarQueue::ctr, in words: queued pixels, chunk indices taken, odd pixels,
// stored ranges, wide entries, tree entries, odd chunks.
constexpr int kCtrQueued = 0, kCtrChunks = 32, kCtrOdd = 64, kCtrRanges = 96, kCtrWide = 128, kCtrTree = 160,
              kCtrOddChunks = 192;
constexpr int kStarCtrWords = 224;
// Pixel classes: no star inside (all taps zero, none stored), taps written by
// star_few / star_map_odd, taps written from the chunks.
constexpr uint8_t kDark = 0, kFew = 1, kQueued = 2;

// All candidates of a pixel in order, into acc (the reference's loop),
// kLightStars at a time: those of the window that lie inside are collected
// into this thread's LDS slots `cand`, then traced, so that a wave runs the
// splat as often as its fullest pixel has stars inside, and the kernel holds
// one copy of it whichever of the tree or the bins lists the candidates.
template <int STEP, bool ODD>
__device__ __forceinline__ void star_seq(const StarPix& P, const SceneK& s, int count, int* cand,
                                         float (&acc)[(2 * STEP + 1) * (2 * STEP + 1)][3]) {
    const float* pos = P.picheck ? s.star_pos : s.bin_pos;
    const float* mag = P.picheck ? s.star_mag : s.bin_mag;
    for (int w = 0; w < count; w += kLightStars) {
        int nq = 0, g = 0;
        for_ranges(P, s, [&](int b, int e) {
            const int len = e - b;
            if (g + len > w && g < w + kLightStars) {
                const int q0 = b + max(0, w - g), q1 = b + min(len, w + kLightStars - g);
                for (int q = q0; q < q1; q++) {
                    float st, sp;
                    if (star_test(P, pos, q, st, sp)) cand[nq++] = q;
                }
            }
            g += len;
        });
        for (int k = 0; k < nq; k++) star_accumulate<STEP, ODD>(P, pos, mag, cand[k], acc);
    }
}

// A pixel's taps lie side by side: taps[ij * NT + tap * 3 + c].  Few pixels
// hold any, and one line then serves a neighbour's three colours (and a
// store) where planes per tap value would take three (27).
template <int STEP>
__device__ __forceinline__ void store_taps(float* taps, size_t ij,
                                           const float (&acc)[(2 * STEP + 1) * (2 * STEP + 1)][3]) {
    constexpr int NT = (2 * STEP + 1) * (2 * STEP + 1) * 3;
#pragma unroll
    for (int t = 0; t < NT; t++) taps[ij * NT + t] = acc[t / 3][t % 3];
}

// Bin rows a lane of star_scan walks itself; taller quads go to star_wide.
constexpr int kScanRows = 4;
// Tiles of 16 x 16 pixels side by side per workgroup of star_scan, at most.
// One in small frames (at 320 x 180 four leave three quarters of the SIMDs
// without a wave: 37 us against 16), kScanTiles from a million pixels on
// (whole frames of three grids with one and with four, us: 1920x1080 588, 836,
// 640 and 591, 842, 638).
constexpr int kScanTiles = 4;

// Sorts the pixels by how much star work they hold: none (most of a frame),
// few candidates with a star inside (kFew), or more than kLightStars
// candidates (kQueued, cut into chunks).  Geometry and inside tests only: the
// lensing's FP64 trigonometry and the splats, which a few percent of the
// pixels need, run on full waves in the kernels below instead of on a few
// lanes of every wave here.  The 2 x kScanRows bin bounds of a pixel load
// together.  Quads taller than kScanRows bin rows and quads across
// phi = 2 pi take a queue entry and are counted by star_wide.  The queue
// entries of the workgroup are staged in LDS and appended with one atomic
// per list: a shared counter takes an atomic only every few nanoseconds.
// (One lane doing all of it, lensing and splats included, took 307 us of a
// 1080p frame and 990 us of a 4K one beside the sky pass.)
__global__ __launch_bounds__(256) void star_scan(const float* thphi, const uint8_t* bh, SceneK s, Cam7 cam, int W,
                                                 int H, float offset, StarQueue Q, int tiles) {
    __shared__ uint32_t s_pix[256 * kScanTiles], s_cnt[256 * kScanTiles];
    __shared__ uint16_t s_wide[256 * kScanTiles], s_tree[256 * kScanTiles];
    __shared__ unsigned s_n[3], s_base[3];
    const unsigned tid = threadIdx.y * 16 + threadIdx.x;
    if (tid < 3) s_n[tid] = 0;
    __syncthreads();
    const int i = blockIdx.y * 16 + threadIdx.y;
    const unsigned lane = __lane_id();
    for (int tile = 0; tile < tiles; tile++) {
        const int j = (blockIdx.x * tiles + tile) * 16 + threadIdx.x;
        const bool valid = i < H && j < W;
        const size_t ij = valid ? (size_t)i * W + j : 0;
        uint8_t cls = kDark;
        bool wide = false, tree = false;
        int count = 0;
        if (valid && bh[ij] == 0) {
            StarPix P;
            star_pixel_geom(thphi, W, i, j, offset, cam, P);
            const int r0 = bin_of(P.mn[0], kBinDT, kBinT), r1 = bin_of(P.mx[0], kBinDT, kBinT);
            const int p0 = bin_of(P.mn[1], kBinDP, kBinP), p1 = bin_of(P.mx[1], kBinDP, kBinP);
            tree = P.picheck;
            wide = !tree && r1 - r0 >= kScanRows;
            if (!tree && !wide) {
                EdgeLines L;
                L.set(P);
                int b[kScanRows], e[kScanRows];
#pragma unroll
                for (int k = 0; k < kScanRows; k++) row_bounds(P, L, s, r0 + k, r1, p0, p1, b[k], e[k]);
#pragma unroll
                for (int k = 0; k < kScanRows; k++) count += e[k] - b[k];
                if (count > kLightStars) {
                    cls = kQueued;
                } else if (count > 0) {
#pragma unroll
                    for (int k = 0; k < kScanRows; k++)
                        for (int q = b[k]; q < e[k]; q++) {
                            float st, sp;
                            if (star_test(P, s.bin_pos, q, st, sp)) cls = kFew;
                        }
                }
            }
        }
        const bool take = cls == kQueued || wide || tree;
        const unsigned long long m = __ballot(take);
        if (m) {
            unsigned pos = 0;
            if (lane == 0) pos = atomicAdd(&s_n[0], (unsigned)__popcll(m));
            pos = __shfl(pos, 0) + (unsigned)__popcll(m & ((1ull << lane) - 1));
            if (take) {
                s_pix[pos] = (uint32_t)ij;
                s_cnt[pos] = wide || tree ? 0u : (uint32_t)count;
                if (wide) s_wide[atomicAdd(&s_n[1], 1u)] = (uint16_t)pos;
                if (tree) s_tree[atomicAdd(&s_n[2], 1u)] = (uint16_t)pos;
            }
        }
        if (valid) Q.lit[ij] = cls;
    }
    __syncthreads();
    if (tid < 3 && s_n[tid])
        s_base[tid] = atomicAdd(&Q.ctr[tid == 0 ? kCtrQueued : tid == 1 ? kCtrWide : kCtrTree], s_n[tid]);
    __syncthreads();
    const unsigned n = s_n[0], qb = s_base[0];
    for (unsigned k = tid; k < n; k += 256) {
        Q.pix[qb + k] = s_pix[k];
        Q.cnt[qb + k] = s_cnt[k];
    }
    for (unsigned k = tid; k < s_n[1]; k += 256) Q.wide[s_base[1] + k] = qb + s_wide[k];
    const size_t last = (size_t)W * H + 63;
    for (unsigned k = tid; k < s_n[2]; k += 256) Q.wide[last - (s_base[2] + k)] = qb + s_tree[k];
}

// Quads across phi = 2 pi per wave of star_wide, at most, and their listed
// tree nodes kept in LDS.  Lanes of one wave part at every node of their
// walks, so a wave of 64 walks takes twice as long as one of 8, and a frame
// has a few hundred to a few thousand such quads: one a wave until every
// SIMD has one, then more.
constexpr int kTreeLanes = 8, kTreeNodes = 512;

// Counts the candidates of the queue entries star_scan left open: a pixel of
// more than kLightStars keeps its entry; one of fewer is kFew if a star is
// inside, else kDark.  One wave per workgroup.  The first `ntree` workgroups
// take the quads across phi = 2 pi, a few lanes each with a quad, and store their listed
// node ranges.  A walk of the star tree is a chain of a few hundred
// dependent steps: it reads the tree from LDS and keeps the listed nodes
// there, so that it runs once (two walks over memory took 150 us of every
// frame, however small).  The other workgroups take tall quads,
// sixteen lanes each with a bin row (most span 5 to 16, a strongly lensed one
// up to all 256).
__global__ __launch_bounds__(64) void star_wide(const float* thphi, SceneK s, Cam7 cam, int W, int H, float offset,
                                                StarQueue Q, unsigned ntree) {
    __shared__ int32_t s_tree[2048];
    __shared__ uint16_t s_node[kTreeNodes][kTreeLanes];
    const unsigned lane = threadIdx.x;
    StarPix P;
    if (blockIdx.x < ntree) {
        const unsigned n = Q.ctr[kCtrTree];
        const unsigned per = min((unsigned)kTreeLanes, (n + ntree - 1) / ntree);   // quads a wave walks at a time
        if (per == 0 || blockIdx.x * per >= n) return;
        const int nodes = (1 << (s.tree_level + 1)) - 1;   // tree_level <= 10
        for (int k = (int)lane; k < nodes; k += 64) s_tree[k] = s.tree[k];
        __syncthreads();
        const size_t last = (size_t)W * H + 63;
        for (unsigned e0 = blockIdx.x * per; e0 < n; e0 += ntree * per) {
            const bool live = lane < per && e0 + lane < n;
            unsigned k = 0, nrng = 0;
            uint32_t ij = 0;
            int count = 0;
            if (live) {
                k = Q.wide[last - (e0 + lane)];
                ij = Q.pix[k];
                star_pixel_geom(thphi, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, cam, P);
                search_tree(s_tree, s.tree_level, P.mn, P.mx, [&](int node) {
                    int b, e;
                    node_range(s_tree, node, b, e);
                    count += e - b;
                    if (nrng < (unsigned)kTreeNodes) s_node[nrng][lane] = (uint16_t)node;
                    nrng++;
                });
            }
            // f(begin, end) for the listed nodes in list order
            auto listed = [&](auto&& f) {
                if (nrng <= (unsigned)kTreeNodes) {
                    for (unsigned x = 0; x < nrng; x++) {
                        int b, e;
                        node_range(s_tree, s_node[x][lane], b, e);
                        f(b, e);
                    }
                } else {
                    search_tree(s_tree, s.tree_level, P.mn, P.mx, [&](int node) {
                        int b, e;
                        node_range(s_tree, node, b, e);
                        f(b, e);
                    });
                }
            };
            const bool few = live && count <= kLightStars;
            if (few && count > 0) {
                bool inside = false;
                listed([&](int b, int e) {
                    for (int q = b; q < e; q++) {
                        float st, sp;
                        if (star_test(P, s.star_pos, q, st, sp)) inside = true;
                    }
                });
                if (inside) Q.lit[ij] = kFew;
            }
            // room for the ranges, one reservation per wave
            const unsigned want = live && !few ? nrng : 0u;
            unsigned inc = want;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const unsigned o = __shfl_up(inc, off);
                if ((int)lane >= off) inc += o;
            }
            const unsigned tot = __shfl(inc, 63);
            unsigned base = 0;
            if (lane == 0 && tot) base = atomicAdd(&Q.ctr[kCtrRanges], tot);
            const unsigned long long r0 = (unsigned long long)__shfl(base, 0) + inc - want;
            if (want) {
                if (r0 + want <= Q.rcap) {
                    unsigned r = (unsigned)r0;
                    listed([&](int b, int e) { Q.ranges[r++] = make_int2(b, e); });
                    Q.rbase[k] = (uint32_t)r0;
                    Q.nnode[k] = want;
                    Q.cnt[k] = (uint32_t)count | kTreePixel;
                    Q.lit[ij] = kQueued;
                } else {
                    Q.lit[ij] = kFew;   // no room: traced by one lane
                }
            }
        }
        return;
    }
    const unsigned n = Q.ctr[kCtrWide];
    const unsigned sub = lane & 15, grp = lane >> 4;
    for (unsigned w0 = (blockIdx.x - ntree) * 4; w0 < n; w0 += (gridDim.x - ntree) * 4) {
        const bool live = w0 + grp < n;
        const unsigned k = live ? Q.wide[w0 + grp] : 0u;
        const uint32_t ij = live ? Q.pix[k] : 0u;
        int r0 = 0, r1 = -1, p0 = 0, p1 = -1;
        EdgeLines L;
        if (live) {
            star_pixel_geom(thphi, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, cam, P);
            r0 = bin_of(P.mn[0], kBinDT, kBinT);
            r1 = bin_of(P.mx[0], kBinDT, kBinT);
            p0 = bin_of(P.mn[1], kBinDP, kBinP);
            p1 = bin_of(P.mx[1], kBinDP, kBinP);
            L.set(P);
        }
        int count = 0;
        for (int r = r0 + (int)sub; r <= r1; r += 16) {
            int b, e;
            row_bounds(P, L, s, r, r1, p0, p1, b, e);
            count += e - b;
        }
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) count += __shfl_xor(count, off);
        bool inside = false;
        if (count > 0 && count <= kLightStars)
            for (int r = r0 + (int)sub; r <= r1; r += 16) {
                int b, e;
                row_bounds(P, L, s, r, r1, p0, p1, b, e);
                for (int q = b; q < e; q++) {
                    float st, sp;
                    if (star_test(P, s.bin_pos, q, st, sp)) inside = true;
                }
            }
        const bool hit = (__ballot(inside) >> (16 * grp) & 0xffffull) != 0;
        if (live && sub == 0) {
            if (count > kLightStars) {
                Q.cnt[k] = (uint32_t)count;
                Q.lit[ij] = kQueued;
            } else if (hit) {
                Q.lit[ij] = kFew;
            }
        }
    }
}

// One lane per queued pixel: its lensing, and its chunk indices.
__global__ __launch_bounds__(256) void star_assign(const float* thphi, SceneK s, Cam7 cam, int W, int H, float offset,
                                                   int lr, const float* area, const float* view, StarQueue Q) {
    const unsigned n = Q.ctr[kCtrQueued];
    const unsigned lane = threadIdx.x & 63;
    for (unsigned e0 = (blockIdx.x * blockDim.x + threadIdx.x) & ~63u; e0 < n; e0 += gridDim.x * blockDim.x) {
        const unsigned k = e0 + lane;
        const uint32_t qc = k < n ? Q.cnt[k] : 0u;
        const unsigned nchunk = queued_chunks(qc);
        unsigned inc = nchunk;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const unsigned o = __shfl_up(inc, off);
            if ((int)lane >= off) inc += o;
        }
        const unsigned tot = __shfl(inc, 63);
        unsigned base = 0;
        if (lane == 0 && tot) base = atomicAdd(&Q.ctr[kCtrChunks], tot);
        base = __shfl(base, 0);
        if (nchunk == 0) continue;
        const uint32_t ij = Q.pix[k];
        const int i = (int)(ij / (uint32_t)W), j = (int)(ij % (uint32_t)W);
        StarPix P;
        star_pixel_geom(thphi, W, i, j, offset, cam, P);
        star_lens(W, ij, i * (W + 1) + j, lr, area, view, cam, P);
        Q.lens[3 * k] = P.frac;
        Q.lens[3 * k + 1] = P.redshft;
        Q.lens[3 * k + 2] = P.red;
        const unsigned long long c0 = (unsigned long long)base + inc - nchunk;
        Q.cstart[k] = (uint32_t)c0;
        if (c0 + nchunk <= Q.cap) {
            const bool odd = star_pixel_odd(P, s);
            unsigned o = 0;
            if (odd) {
                Q.cnt[k] = qc | kOddPixel;
                o = atomicAdd(&Q.ctr[kCtrOddChunks], nchunk);
            }
            for (unsigned c = 0; c < nchunk; c++) {
                Q.owner[c0 + c] = k;
                if (odd) Q.oddc[o + c] = (uint32_t)c0 + c;
            }
        } else {
            // its chunks do not fit: no chunk work, one lane traces it
            Q.cnt[k] = 0;
            Q.lit[ij] = kFew;
            for (unsigned long long c = c0; c < Q.cap && c < c0 + nchunk; c++) Q.owner[c] = kNoOwner;
        }
    }
}

// Pixels per workgroup of star_few, at most: a span of the frame is chosen so
// that there are about a thousand workgroups (few_span), each gathering
// enough kFew pixels to fill its waves where the frame is large.
constexpr int kFewSpan = 8192;

// The kFew pixels of a span of the frame, gathered in LDS so that full waves
// trace them, one pixel per lane: all its candidates in order.
template <int STEP>
__global__ __launch_bounds__(256) void star_few(const float* thphi, const uint8_t* bh, SceneK s, Cam7 cam, int W,
                                                int H, float offset, int lr, const float* area, const float* view,
                                                float* taps, StarQueue Q, int span) {
    constexpr int FW = 2 * STEP + 1;
    __shared__ int s_cand[256][kLightStars];
    __shared__ uint16_t s_list[kFewSpan];
    __shared__ unsigned s_n;
    const size_t NP = (size_t)W * H;
    const size_t p0 = (size_t)blockIdx.x * span;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    for (int k = 0; k < span; k += 256) {
        const size_t p = p0 + k + threadIdx.x;
        if (p < NP && Q.lit[p] == kFew) s_list[atomicAdd(&s_n, 1u)] = (uint16_t)(k + threadIdx.x);
    }
    __syncthreads();
    const unsigned n = s_n;
    for (unsigned t = threadIdx.x; t < n; t += 256) {
        const size_t ij = p0 + s_list[t];
        StarPix P;
        star_pixel(thphi, bh, W, (int)(ij / (size_t)W), (int)(ij % (size_t)W), offset, lr, area, view, cam, P);
        const bool odd = star_pixel_odd(P, s);
        wave_append(Q.odd, &Q.ctr[kCtrOdd], odd, (uint32_t)ij);
        if (odd) continue;
        float acc[FW * FW][3];
#pragma unroll
        for (int u = 0; u < FW * FW; u++) acc[u][0] = acc[u][1] = acc[u][2] = 0.f;
        int count = 0;
        for_ranges(P, s, [&](int b, int e) { count += e - b; });
        star_seq<STEP, false>(P, s, count, s_cand[threadIdx.x], acc);
        store_taps<STEP>(taps, ij, acc);
    }
}

// One lane per odd pixel (star_pixel_odd) of few candidates: all its
// candidates, each tap checked for the reference's slow expression.
template <int STEP>
__global__ __launch_bounds__(256) void star_map_odd(const float* thphi, const uint8_t* bh, SceneK s, Cam7 cam,
                                                    int W, int H, float offset, int lr, const float* area,
                                                    const float* view, float* taps, StarQueue Q) {
    constexpr int FW = 2 * STEP + 1;
    __shared__ int s_cand[256][kLightStars];
    const unsigned n = Q.ctr[kCtrOdd];
    for (unsigned k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const uint32_t ij = Q.odd[k];
        float acc[FW * FW][3];
#pragma unroll
        for (int u = 0; u < FW * FW; u++) acc[u][0] = acc[u][1] = acc[u][2] = 0.f;
        StarPix P;
        if (star_pixel(thphi, bh, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, lr, area, view,
                       cam, P)) {
            int count = 0;
            for_ranges(P, s, [&](int b, int e) { count += e - b; });
            star_seq<STEP, true>(P, s, count, s_cand[threadIdx.x], acc);
        }
        store_taps<STEP>(taps, ij, acc);
    }
}

// One step of store_tap_sums on the wave's first n values, pairing each lane
// with lane ^ OFF: h = ceil(n / 2) values stay, the lanes whose bit OFF is
// clear keep the first h, the others the rest.
template <int OFF, int N>
__device__ __forceinline__ void fold_taps(float* v, unsigned lane) {
    constexpr int h = (N + 1) / 2;
#pragma unroll
    for (int k = 0; k < h; k++) {
        const float a = v[k], b = h + k < N ? v[h + k] : 0.f;
        if (OFF == 32) {
            const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
            v[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        } else if (OFF == 16) {
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
            v[k] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        } else {
            const bool up = (lane & OFF) != 0;
            v[k] = (up ? b : a) + __shfl_xor(up ? a : b, OFF);
        }
    }
}

// out[t] = the sum over the wave's lanes of value t of acc, in the order of
// the xor butterfly 32, 16, 8, 4, 2, 1.  Each step halves the values a lane
// holds instead of summing all of them on every lane: 29 exchanges for the
// 27 tap values of step 1 instead of 162, with the same pairs added (an
// addition's order within a pair does not matter), so the same sums bit for
// bit.  The two widest steps are the swap instructions of the lane halves
// and of the 16-lane rows, which move both directions of an exchange at
// once.  `any` false: every value is zero.
template <int NT>
__device__ __forceinline__ void store_tap_sums(float (&acc)[NT / 3][3], bool any, float* out, unsigned lane) {
    constexpr int n1 = (NT + 1) / 2, n2 = (n1 + 1) / 2, n3 = (n2 + 1) / 2, n4 = (n3 + 1) / 2, n5 = (n4 + 1) / 2,
                  n6 = (n5 + 1) / 2;
    if (!any) {
        for (unsigned t = lane; t < (unsigned)NT; t += 64) out[t] = 0.f;
        return;
    }
    float v[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) v[t] = acc[t / 3][t % 3];
    fold_taps<32, NT>(v, lane);
    fold_taps<16, n1>(v, lane);
    fold_taps<8, n2>(v, lane);
    fold_taps<4, n3>(v, lane);
    fold_taps<2, n4>(v, lane);
    fold_taps<1, n5>(v, lane);
    // the values this lane is left with: `real` of them from t0 on
    int t0 = 0, real = NT, n = NT;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const int h = (n + 1) / 2;
        if (lane & off) {
            t0 += h;
            real -= h;
        } else {
            real = min(real, h);
        }
        n = h;
    }
#pragma unroll
    for (int k = 0; k < n6; k++)
        if (k < real) out[t0 + k] = v[k];
}

// What star_map_chunk needs of a chunk and its pixel, made by star_heads with
// one lane per chunk (a wave making it for its own chunk spent a fifth of
// its instructions on it) and kept in the chunk's partial until the chunk's
// sums replace it: kHeadWords words, at most the 27 floats of the smallest
// partial.
struct ChunkHead {
    float t[4], p[4];      // the quad's corners
    EdgeLines edge;        // its edges' lines (side: see kHead* for more bits)
    float frac, redshft, red;
    unsigned rows, cols;   // first and last bin row / column (low, high half)
    unsigned g0, g1;       // its candidates [g0, g1) of the pixel's
    unsigned ij, rbase, nrange;
};
constexpr int kHeadWords = sizeof(ChunkHead) / 4;
static_assert(kHeadWords <= 27, "a chunk's head fits its partial");
constexpr unsigned kHeadFlip = 0x100u, kHeadTree = 0x200u, kHeadOne = 0x400u;

template <int NT>
__global__ __launch_bounds__(256) void star_heads(const float* thphi, Cam7 cam, int W, float offset, StarQueue Q) {
    const unsigned nch = min(Q.ctr[kCtrChunks], Q.cap);
    for (unsigned c = blockIdx.x * blockDim.x + threadIdx.x; c < nch; c += gridDim.x * blockDim.x) {
        ChunkHead h;
        const uint32_t k = Q.owner[c];
        const uint32_t qc = k == kNoOwner ? 0u : Q.cnt[k];
        h.g0 = h.g1 = 0;
        if (qc) {
            h.ij = Q.pix[k];
            h.g0 = (c - Q.cstart[k]) * (unsigned)kChunk;
            h.g1 = min(h.g0 + kChunk, queued_count(qc));
            StarPix P;
            star_pixel_geom(thphi, W, (int)(h.ij / (uint32_t)W), (int)(h.ij % (uint32_t)W), offset, cam, P);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                h.t[q] = P.t[q];
                h.p[q] = P.p[q];
            }
            h.edge.set(P);
            const bool tree = (qc & kTreePixel) != 0;
            h.edge.side |= (P.sgn < 0 ? kHeadFlip : 0u) | (tree ? kHeadTree : 0u) |
                           (queued_chunks(qc) == 1 ? kHeadOne : 0u);
            h.frac = Q.lens[3 * k];
            h.redshft = Q.lens[3 * k + 1];
            h.red = Q.lens[3 * k + 2];
            const unsigned r0 = bin_of(P.mn[0], kBinDT, kBinT), r1 = bin_of(P.mx[0], kBinDT, kBinT);
            h.rows = r0 | r1 << 16;
            h.cols = (unsigned)bin_of(P.mn[1], kBinDP, kBinP) | (unsigned)bin_of(P.mx[1], kBinDP, kBinP) << 16;
            h.rbase = tree ? Q.rbase[k] : 0u;
            h.nrange = tree ? Q.nnode[k] : r1 - r0 + 1;
        }
        const unsigned* w = reinterpret_cast<const unsigned*>(&h);
        unsigned* o = reinterpret_cast<unsigned*>(Q.partial + (size_t)c * NT);
        if (h.g1)
#pragma unroll
            for (int q = 0; q < kHeadWords; q++) o[q] = w[q];
        // The two instances of star_map_chunk run side by side, and each
        // replaces the heads of its chunks by their sums: which instance owns
        // a chunk must not be read from its head.
        if (qc == 0 || (qc & kOddPixel)) Q.owner[c] = kNoOwner;
    }
}

// Inclusive sum over the wave's lanes: DPP row shifts, then the rows' last
// lanes broadcast to the rows after them.
__device__ __forceinline__ unsigned wave_scan(unsigned v) {
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   // row_bcast15 into rows 1, 3
    v += (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   // row_bcast31 into rows 2, 3
    return v;
}

// One wavefront per chunk (grid-stride): lane l takes the chunk's
// candidates l, l + 64, ...; the taps are reduced over the wave in a fixed
// order into the chunk's partial, summed per pixel by star_chunk_reduce.
// The wave walks the candidate ranges its head names (bin rows, or stored
// tree ranges) 64 at a time: each lane loads one range, a wave scan gives the
// ranges' first candidate numbers (kept in LDS), and each lane finds the
// range of each of its candidates.
template <int STEP, bool ODD>
__global__ __launch_bounds__(256) void star_map_chunk(SceneK s, Cam7 cam, float* taps, StarQueue Q) {
    constexpr int FW = 2 * STEP + 1;
    constexpr int NT = FW * FW * 3;
    const unsigned lane = threadIdx.x & 63;
    const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    const unsigned nwaves = (gridDim.x * blockDim.x) >> 6;
    const unsigned nch = ODD ? Q.ctr[kCtrOddChunks] : min(Q.ctr[kCtrChunks], Q.cap);
    __shared__ int s_beg[4][64];
    __shared__ unsigned s_pre[4][65];
    // stars found inside, staged until 64 can be splatted by a full wave
    __shared__ int s_iq[4][128];
    __shared__ float s_ist[4][128], s_isp[4][128];
    const unsigned wslot = threadIdx.x >> 6;
    for (unsigned x = wave; x < nch; x += nwaves) {
        const unsigned c = ODD ? Q.oddc[x] : x;
        if (!ODD && Q.owner[c] == kNoOwner) continue;   // no work, or the other instance's (oddc lists those)
        // the head, one word per lane, spread to scalars
        ChunkHead h;
        {
            float* part = Q.partial + (size_t)c * NT;
            const int w = lane < (unsigned)kHeadWords ? __float_as_int(part[lane]) : 0;
            int* o = reinterpret_cast<int*>(&h);
#pragma unroll
            for (int q = 0; q < kHeadWords; q++) o[q] = __builtin_amdgcn_readlane(w, q);
        }
        const uint32_t ij = h.ij;
        const unsigned g0 = h.g0, g1 = h.g1;
        const bool tree = (h.edge.side & kHeadTree) != 0;
        StarPix P;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            P.t[q] = h.t[q];
            P.p[q] = h.p[q];
        }
        P.colours = cam.colours;
        P.mn[1] = fminf(fminf(P.p[0], P.p[1]), fminf(P.p[2], P.p[3]));
        P.mx[1] = fmaxf(fmaxf(P.p[0], P.p[1]), fmaxf(P.p[2], P.p[3]));
        P.frac = h.frac;
        P.redshft = h.redshft;
        P.red = h.red;
        P.sgn = h.edge.side & kHeadFlip ? -1 : 1;
        P.picheck = tree;   // a quad across phi = 2 pi
        const float* pos = tree ? s.star_pos : s.bin_pos;
        const float* mag = tree ? s.star_mag : s.bin_mag;
        float acc[FW * FW][3];
#pragma unroll
        for (int u = 0; u < FW * FW; u++) acc[u][0] = acc[u][1] = acc[u][2] = 0.f;
        bool any = false;
        {
            // The pixel's candidate ranges, 64 at a time: the stored tree
            // node ranges, or the bin rows r0..r1 cut to their phi spans.
            // Candidates are tested one per lane; the stars inside are
            // staged in LDS and splatted 64 at a time, so that the long
            // splat runs on full waves however few candidates pass.  One
            // loop alternates filling (up to 64 staged) and splatting, so
            // that the splat has one call site.
            const int r0 = (int)(h.rows & 0xffffu), r1 = (int)(h.rows >> 16);
            const int p0 = (int)(h.cols & 0xffffu), p1 = (int)(h.cols >> 16);
            const int nrange = (int)h.nrange;
            // `any`: a star was found inside.
            // wave-uniform state: current block, its candidate window
            // [gb, a1), the candidates before it, staged stars
            int kb = 0;
            unsigned base = 0, tot = 0, gb = 0, a1 = 0, nin = 0;
            bool loaded = false, done = false;
            int row = 0;   // per lane: range of the block holding its next candidate
            while (true) {
                while (!done && nin < 64) {
                    if (!loaded) {
                        if (kb >= nrange || base >= g1) {
                            done = true;
                            break;
                        }
                        const int k = kb + (int)lane;
                        int b = 0, e = 0;
                        if (k < nrange) {
                            if (tree) {
                                const int2 R = Q.ranges[h.rbase + (unsigned)k];
                                b = R.x;
                                e = R.y;
                            } else {
                                const int r = r0 + k;
                                row_bounds(P, h.edge, s, r, r1, p0, p1, b, e);
                            }
                        }
                        const unsigned inc = wave_scan((unsigned)(e - b));
                        __builtin_amdgcn_wave_barrier();
                        s_beg[wslot][lane] = b;
                        s_pre[wslot][lane + 1] = inc;
                        if (lane == 0) s_pre[wslot][0] = 0;
                        tot = (unsigned)__builtin_amdgcn_readlane((int)inc, 63);
                        __builtin_amdgcn_wave_barrier();
                        gb = max(base, g0);
                        a1 = min(base + tot, g1);
                        // range k with s_pre[k] <= x < s_pre[k+1] for the
                        // lane's first candidate, by bisection; later ones
                        // walk on from it (x grows)
                        row = 0;
                        if (gb + lane < a1) {
                            const unsigned x = gb + lane - base;
                            int hi2 = 63;
                            while (row < hi2) {
                                int mid = (row + hi2 + 1) >> 1;
                                if (s_pre[wslot][mid] <= x) row = mid;
                                else hi2 = mid - 1;
                            }
                        }
                        loaded = true;
                    }
                    if (gb >= a1) {
                        base += tot;
                        kb += 64;
                        loaded = false;
                        continue;
                    }
                    const unsigned g = gb + lane;
                    bool in = false;
                    int q = 0;
                    float st = 0.f, sp = 0.f;
                    if (g < a1) {
                        const unsigned x = g - base;   // candidate number within this block
                        while (s_pre[wslot][row + 1] <= x) row++;
                        q = s_beg[wslot][row] + (int)(x - s_pre[wslot][row]);
                        in = star_test(P, pos, q, st, sp);
                    }
                    const unsigned long long m = __ballot(in);
                    if (in) {
                        const unsigned k = nin + (unsigned)__popcll(m & ((1ull << lane) - 1));
                        s_iq[wslot][k] = q;
                        s_ist[wslot][k] = st;
                        s_isp[wslot][k] = sp;
                    }
                    nin += (unsigned)__popcll(m);
                    gb += 64;
                    __builtin_amdgcn_wave_barrier();
                }
                if (nin == 0) break;
                any = true;
                const unsigned take = nin < 64 ? nin : 64u;
                if (lane < take)
                    star_splat<STEP, ODD>(P, mag, s_iq[wslot][lane], s_ist[wslot][lane], s_isp[wslot][lane],
                                          acc);
                const unsigned rest = nin - take;
                int q2 = 0;
                float st2 = 0.f, sp2 = 0.f;
                if (lane < rest) {
                    q2 = s_iq[wslot][64 + lane];
                    st2 = s_ist[wslot][64 + lane];
                    sp2 = s_isp[wslot][64 + lane];
                }
                __builtin_amdgcn_wave_barrier();
                if (lane < rest) {
                    s_iq[wslot][lane] = q2;
                    s_ist[wslot][lane] = st2;
                    s_isp[wslot][lane] = sp2;
                }
                nin = rest;
                __builtin_amdgcn_wave_barrier();
                if (done && nin == 0) break;
            }
        }
        // the sums over the lanes: straight into the taps for a pixel of one
        // chunk, else into the chunk's partial for star_chunk_reduce
        const bool one = (h.edge.side & kHeadOne) != 0;
        store_tap_sums<NT>(acc, any, one ? taps + (size_t)ij * NT : Q.partial + (size_t)c * NT, lane);
    }
}

// The queued pixels of several chunks: their partials summed in chunk order,
// one thread per (pixel, tap value), eight partials in flight at a time (a
// pixel may have hundreds).  A pixel of one chunk is its partial, which
// star_map_chunk stores itself.
template <int STEP>
__global__ __launch_bounds__(256) void star_chunk_reduce(float* taps, StarQueue Q) {
    constexpr int NT = (2 * STEP + 1) * (2 * STEP + 1) * 3;
    const unsigned n = Q.ctr[kCtrQueued];
    const size_t total = (size_t)n * NT;
    for (size_t x = (size_t)blockIdx.x * blockDim.x + threadIdx.x; x < total; x += (size_t)gridDim.x * blockDim.x) {
        const unsigned k = (unsigned)(x / NT), t = (unsigned)(x % NT);
        const unsigned nchunk = queued_chunks(Q.cnt[k]);
        if (nchunk <= 1) continue;   // 0: traced by one lane
        const float* part = Q.partial + (size_t)Q.cstart[k] * NT + t;
        float v = 0.f;
        unsigned ch = 0;
        for (; ch + 8 <= nchunk; ch += 8) {
            float y[8];
#pragma unroll
            for (int u = 0; u < 8; u++) y[u] = part[(size_t)(ch + u) * NT];
#pragma unroll
            for (int u = 0; u < 8; u++) v += y[u];
        }
        for (; ch < nchunk; ch++) v += part[(size_t)ch * NT];
        taps[(size_t)Q.pix[k] * NT + t] = v;
    }
}

// Column j of a frame that wraps around, for j in [-W, 2 W) at least.
__device__ __forceinline__ int wrap_frame(int j, int W) {
    while (j < 0) j += W;
    while (j >= W) j -= W;
    return j;
}

// makePix (MakeImageKernel.cu:802-835) of one pixel's summed star light.
__device__ __forceinline__ void make_pix(float br, float bg, float bb, uint8_t* img, size_t ij) {
    if (br == 0.f && bg == 0.f && bb == 0.f) {   // most of a frame
        reinterpret_cast<uchar4*>(img)[ij] = make_uchar4(0, 0, 0, 255);
        return;
    }
    float r = sqrtf(br), g = sqrtf(bg), b = sqrtf(bb);
    float mxc = fmaxf(fmaxf(r, g), b);
    if (mxc > 255.f) {
        float hh, ss, pp;
        rgb_to_hsp(r / 255.f, g / 255.f, b / 255.f, hh, ss, pp);
        pp = 1.0f;
        hsp_to_rgb(hh, ss, pp, r, g, b);
        r *= 255;
        g *= 255;
        b *= 255;
    }
    uchar4 o;
    o.x = (uint8_t)min(255, cvt_i32(b + 0.f));
    o.y = (uint8_t)min(255, cvt_i32(g + 0.f));
    o.z = (uint8_t)min(255, cvt_i32(r + 0.f));
    o.w = 255;
    reinterpret_cast<uchar4*>(img)[ij] = o;
}

// sumStarLight (MakeImageKernel.cu:753-773) + makePix; trail (or null): the
// frame's star trails, added after the taps (factor 1).
// sumStarLight (MakeImageKernel.cu:753-773, bounds-checked) + makePix (:802-835)
template <int STEP>
__global__ __launch_bounds__(256) void star_sum(const float* taps, const uint8_t* lit, int W, int H, uint8_t* img,
                                                float* o_star, const float* trail) {
    constexpr int FW = 2 * STEP + 1;
    constexpr int NT = FW * FW * 3;
    constexpr int TW = 16 + 2 * STEP;
    // the tile's classes with its border; a row outside the frame is dark
    __shared__ uint8_t s_lit[TW][TW];
    const int i0 = blockIdx.y * 16 - STEP, j0 = blockIdx.x * 16 - STEP;
    for (int c = threadIdx.y * 16 + threadIdx.x; c < TW * TW; c += 256) {
        const int ii = i0 + c / TW;
        const int jj = wrap_frame(j0 + c % TW, W);
        s_lit[c / TW][c % TW] = ii >= 0 && ii < H ? lit[(size_t)ii * W + jj] : kDark;
    }
    __syncthreads();
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= H || j >= W) return;
    float br = 0.f, bg = 0.f, bb = 0.f;
    const float factor = 20.f;
    // a row of neighbours at a time: their taps are in flight together, and
    // added in order (a dark neighbour's are zero and not stored)
#pragma unroll
    for (int u = 0; u < FW; u++) {
        bool any = false;
#pragma unroll
        for (int v = 0; v < FW; v++) any = any || s_lit[threadIdx.y + u][threadIdx.x + v] != kDark;
        if (!any) continue;
        float3 x[FW];
#pragma unroll
        for (int v = 0; v < FW; v++) {
            x[v] = make_float3(0.f, 0.f, 0.f);
            if (s_lit[threadIdx.y + u][threadIdx.x + v] != kDark) {
                const size_t src = (size_t)(i + u - STEP) * W + wrap_frame(j + v - STEP, W);
                const float* t = taps + src * NT + 3 * (FW * FW - (FW * u + v + 1));
                x[v] = make_float3(t[0], t[1], t[2]);
            }
        }
#pragma unroll
        for (int v = 0; v < FW; v++) {
            br += factor * x[v].x;
            bg += factor * x[v].y;
            bb += factor * x[v].z;
        }
    }
    const size_t ij = (size_t)i * W + j;
    if (trail) {
        br += trail[3 * ij];
        bg += trail[3 * ij + 1];
        bb += trail[3 * ij + 2];
    }
    if (o_star) {
        o_star[3 * ij] = br;
        o_star[3 * ij + 1] = bg;
        o_star[3 * ij + 2] = bb;
    }
    make_pix(br, bg, bb, img, ij);
}

// ---- star trails and diffraction (MakeImageKernel.cu:98-174,517-537,
// 618-629,775-800): effects of a sequence of frames.
//
// Each frame records, per star, the pixels its images land in (pixels with
// fewer than S/100 candidate stars in their tree leaves), keeping the first
// kTrailNum; the next frame draws, for each image, a fading line from the
// previous frame's image of the same star that lies closest to the
// direction of celestial motion (the gradient field rotated by 90 degrees),
// within 45 degrees and M/25 pixels, unless the star moved by at most one
// pixel.  The reference appends images in atomic order and its lines
// overwrite each other in whatever order threads run; here a star's images
// are kept in pixel order and overlapping trails keep the per-channel
// maximum, so a frame does not depend on scheduling.

__global__ __launch_bounds__(256) void trail_clear(TrailK T, int frame0, size_t n3) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t q = t; q < (size_t)T.S; q += stride) {
        T.nhits[q] = 0;
        T.count[(size_t)T.cur * T.S + q] = 0;
        if (frame0) T.count[(size_t)(1 - T.cur) * T.S + q] = 0;
    }
    for (size_t p = t; p < n3; p += stride) T.trail[p] = 0.f;
    if (t == 0) T.stats[1] = 0;
}

// makeGradField (MakeImageKernel.cu:517-537) per pixel corner.  Corners in
// the shadow get (0, 0) (the reference leaves them unwritten), and the
// right-hand neighbour of the last corner of the last row, which the
// reference reads one element past its array, counts as invalid.
__global__ __launch_bounds__(256) void trail_grad(const float* thphi, int W, int H, float* grad) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i > H || j > W) return;
    const int M1 = W + 1;
    const size_t NC = (size_t)M1 * (H + 1);
    auto th = [&](size_t c) { return c < NC ? thphi[2 * c] : -1.f; };
    const float up = th((size_t)min(H, i + 1) * M1 + j);
    const float down = th((size_t)max(0, i - 1) * M1 + j);
    const float left = th((size_t)i * M1 + max(0, j - 1));
    const float right = th((size_t)i * M1 + min(M1, j + 1));
    const float mid = th((size_t)i * M1 + j);
    float gx = 0.f, gy = 0.f;
    if (mid > 0) {
        float xdir = 0;
        if (up > 0 && down > 0) xdir = .5f * (up - mid) - .5f * (down - mid);
        float ydir = 0;
        if (left > 0 && right > 0) ydir = .5f * (right - mid) - .5f * (left - mid);
        gx = -ydir;
        gy = xdir;
    }
    grad[2 * ((size_t)i * M1 + j)] = gx;
    grad[2 * ((size_t)i * M1 + j) + 1] = gy;
}

// One image: star q of the scene in pixel pix.  The first kTrailHits images of a
// star that are found take a slot each, the others (few stars have so many) a
// place in the list that trail_over goes through.
__device__ __forceinline__ void trail_record(const TrailK& T, int q, uint32_t pix) {
    const unsigned slot = atomicAdd(&T.nhits[q], 1u);
    if (slot < (unsigned)kTrailHits) {
        T.hit_pix[(size_t)q * kTrailHits + slot] = pix;
        return;
    }
    const unsigned at = atomicAdd(&T.stats[1], 1u);
    if (at < (unsigned)T.S * kTrailHits) T.over[at] = make_int2(q, (int)pix);
}

// Largest star tree (level 10), held in LDS for the walks.
constexpr int kTreeWords = (1 << 11) - 1;

// Whether the pixel's starsToCheck (MakeImageKernel.cu:273-282) stays below
// S/100: the walk of the star tree ends once it does not.
__device__ bool trail_pixel(const SceneK& s, const StarPix& P) {
    int starsToCheck = 0;
    search_tree_until(
        s.tree, s.tree_level, P.mn, P.mx,
        [&](int node) {
            int b, e;
            node_range(s.tree, node, b, e);
            starsToCheck += e - b;
        },
        [&] { return starsToCheck >= s.S / 100; });
    return starsToCheck < s.S / 100;
}

// The images among candidates b + first, b + first + step, .. below e: as in
// the star pass, binned stars, or tree order for quads across phi = 2 pi.
__device__ __forceinline__ void trail_range(const TrailK& T, const SceneK& s, const StarPix& P, uint32_t ij, int b,
                                            int e, int first, int step) {
    const float* pos = P.picheck ? s.star_pos : s.bin_pos;
    for (int k = b + first; k < e; k += step) {
        float st, sp;
        if (star_test(P, pos, k, st, sp)) trail_record(T, P.picheck ? k : s.bin_idx[k], ij);
    }
}

// The images of this frame: per pixel with starsToCheck < S/100
// (MakeImageKernel.cu:273-282,301), every star inside its quad.  Runs after the
// star pass has sorted the pixels: one that is kDark has no star inside.
// trail_hits does the kFew pixels, gathered in LDS from a span of the frame so
// that full waves walk the star tree (from LDS); trail_queued the queued ones,
// sixteen lanes to a pixel's candidates.  Most pixels hold no star: a lane per pixel of the
// frame, walking the tree for each, took 980 us at 1366 x 768 with 100000
// stars.
__global__ __launch_bounds__(256) void trail_hits(const float* thphi, SceneK s, Cam7 cam, int W, int H, float offset,
                                                  TrailK T, const uint8_t* lit, int span) {
    __shared__ int32_t s_tree[kTreeWords];
    __shared__ uint16_t s_list[kFewSpan];
    __shared__ unsigned s_n;
    const size_t NP = (size_t)W * H;
    const size_t p0 = (size_t)blockIdx.x * span;
    const int words = (2 << s.tree_level) - 1;
    if (threadIdx.x == 0) s_n = 0;
    for (int k = threadIdx.x; k < words; k += 256) s_tree[k] = s.tree[k];
    __syncthreads();
    for (int k = 0; k < span; k += 256) {
        const size_t p = p0 + k + threadIdx.x;
        if (p < NP && lit[p] == kFew) s_list[atomicAdd(&s_n, 1u)] = (uint16_t)(k + threadIdx.x);
    }
    __syncthreads();
    s.tree = s_tree;
    for (unsigned t = threadIdx.x; t < s_n; t += 256) {
        const size_t ij = p0 + s_list[t];
        const int i = (int)(ij / (size_t)W), j = (int)(ij % (size_t)W);
        StarPix P;
        star_pixel_geom(thphi, W, i, j, offset, cam, P);
        if (!trail_pixel(s, P)) continue;
        for_ranges(P, s, [&](int b, int e) { trail_range(T, s, P, (uint32_t)ij, b, e, 0, 1); });
    }
}

__global__ __launch_bounds__(256) void trail_queued(const float* thphi, SceneK s, Cam7 cam, int W, float offset,
                                                    TrailK T, StarQueue Q) {
    __shared__ int32_t s_tree[kTreeWords];
    const int words = (2 << s.tree_level) - 1;
    for (int k = threadIdx.x; k < words; k += 256) s_tree[k] = s.tree[k];
    __syncthreads();
    s.tree = s_tree;
    const unsigned n = Q.ctr[kCtrQueued];
    const unsigned lane = __lane_id(), wave = blockIdx.x * 4 + threadIdx.x / 64;
    StarPix P;
    for (unsigned e0 = wave * 16; e0 < n; e0 += gridDim.x * 4 * 16) {
        bool pass = false;
        if (lane < 16 && e0 + lane < n && Q.cnt[e0 + lane]) {
            const uint32_t ij = Q.pix[e0 + lane];
            star_pixel_geom(thphi, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, cam, P);
            pass = trail_pixel(s, P);
        }
        unsigned todo = (unsigned)__ballot(pass);
        // four of the pixels at a time, sixteen lanes each
        while (todo) {
            unsigned m = todo;
            for (unsigned g = 0; g < lane / 16; g++) m &= m - 1;
            if (m) {
                const unsigned k = e0 + (unsigned)__ffs((int)m) - 1;
                const uint32_t ij = Q.pix[k];
                star_pixel_geom(thphi, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, cam, P);
                for_ranges(P, s, [&](int b, int e) { trail_range(T, s, P, ij, b, e, (int)(lane & 15), 16); });
            }
            for (int g = 0; g < 4; g++) todo &= todo - 1;
        }
    }
}

// The images beyond the slots: each goes round its star's slots, leaves the
// lesser pixel in each and takes the other on, so that a star keeps its first
// images in pixel order, whatever the order they were found in.  Slots only
// ever fall: one read as less or equal is passed over, and what has been all the
// way round is no less than any of them.
__global__ __launch_bounds__(256) void trail_over(TrailK T) {
    const unsigned n = min(T.stats[1], (unsigned)T.S * kTrailHits);
    for (unsigned t = blockIdx.x * 256 + threadIdx.x; t < n; t += gridDim.x * 256) {
        const int2 image = T.over[t];
        uint32_t* hp = T.hit_pix + (size_t)image.x * kTrailHits;
        uint32_t pix = (uint32_t)image.y, v[kTrailHits];
#pragma unroll
        for (int k = 0; k < kTrailHits; k++) v[k] = hp[k];
#pragma unroll
        for (int k = 0; k < kTrailHits; k++)
            if (v[k] > pix) pix = max(pix, atomicMin(&hp[k], pix));
    }
}

// Star q: its first kTrailNum images in pixel order become this frame's cache
// (MakeImageKernel.cu:102-104).
__device__ __forceinline__ void trail_cache(const TrailK& T, int q, int W) {
    const int n = (int)min(T.nhits[q], (unsigned)kTrailHits);
    if (n == 0) return;
    const uint32_t* hp = T.hit_pix + (size_t)q * kTrailHits;
    int2* c = T.cache + ((size_t)T.cur * T.S + q) * kTrailNum;
    for (int k = 0; k < n; k++) {   // a star has a few images
        const uint32_t pix = hp[k];
        int rank = 0;
        for (int m = 0; m < n; m++) rank += hp[m] < pix || (hp[m] == pix && m < k);
        if (rank < kTrailNum) c[rank] = make_int2((int)(pix / (uint32_t)W), (int)(pix % (uint32_t)W));
    }
    T.count[(size_t)T.cur * T.S + q] = min(n, kTrailNum);
}

__device__ __forceinline__ void trail_put(float* trail, size_t ij, float v, int ch) {
    if (v >= 0.f) atomicMax(reinterpret_cast<int*>(trail) + 3 * ij + ch, __float_as_int(v));
}

// addTrails (MakeImageKernel.cu:98-174) for one image of one star; the first
// `ncache` workgroups fill this frame's half of the cache instead, which nothing
// reads before the next frame.
__global__ __launch_bounds__(256) void trail_lines(const float* thphi, SceneK s, TrailK T, Cam7 cam, int W, int H,
                                                   float offset, int lr, const float* area, const float* view,
                                                   unsigned ncache) {
    if (blockIdx.x < ncache) {
        const int q = (int)(blockIdx.x * 256 + threadIdx.x);
        if (q < T.S) trail_cache(T, q, W);
        return;
    }
    const float* grad = T.grad;
    const size_t t = (size_t)(blockIdx.x - ncache) * 256 + threadIdx.x;
    if (t >= (size_t)T.S * kTrailHits) return;
    const int q = (int)(t / kTrailHits), slot = (int)(t % kTrailHits);
    if (slot >= (int)min(T.nhits[q], (unsigned)kTrailHits)) return;
    const size_t h = (size_t)q * kTrailHits + slot;
    const int M = W, M1 = W + 1;
    const uint32_t pix = T.hit_pix[h];
    const int i = (int)(pix / (uint32_t)W), j = (int)(pix % (uint32_t)W);
    const int prev_half = 1 - T.cur;
    const int pc = T.count[(size_t)prev_half * T.S + q];
    const int2* pcache = T.cache + ((size_t)prev_half * T.S + q) * kTrailNum;
    float traildist = (float)M;
    float angle = BT_FPI2;
    int2 prev = make_int2(0, 0);
    bool line = false;
    for (int w = 0; w < pc; w++) {
        const int2 pr = pcache[w];
        const int dx = pr.x - i, dy = pr.y - j;
        const int dxx = dx * dx, dyy = dy * dy;
        if (dxx <= 1 && dyy <= 1) {
            line = false;
            break;
        }
        const float grx = grad[2 * ((size_t)pr.x * M1 + pr.y)], gry = grad[2 * ((size_t)pr.x * M1 + pr.y) + 1];
        const float dist = sqrtf((float)(dxx + dyy));
        if (dist > M / 25.f) continue;
        const float div = (dist * sqrtf(grx * grx + gry * gry));
        const float a1 = f_acos((1.f * dx * grx + 1.f * dy * gry) / div);
        const float a2 = f_acos((1.f * dx * -grx + 1.f * dy * -gry) / div);
        const float a = fminf(a1, a2);
        if (a > angle || a > BT_FPI * .25f) continue;
        if (a < angle) {
            angle = a;
            traildist = dist;
            prev = pr;
            line = true;
        }
    }
    if (!line) return;
    StarPix P;
    star_pixel_geom(thphi, W, i, j, offset, cam, P);
    star_lens(W, pix, i * M1 + j, lr, area, view, cam, P);
    const float2 mg = reinterpret_cast<const float2*>(s.star_mag)[q];
    const float part = mg.x + P.red;
    const float temp = 46.f / P.redshft * ((1.f / ((0.92f * mg.y) + 1.7f)) + (1.f / ((0.92f * mg.y) + 0.62f))) - 10.f;
    const float* col = cam.colours + 6 * max(0, min(cvt_i32(floorf(temp)), 390));
    const int deltax = i - prev.x, deltay = j - prev.y;
    const int sgnDeltaX = deltax < 0 ? -1 : 1, sgnDeltaY = deltay < 0 ? -1 : 1;
    const float deltaerr = deltay == 0 ? fabsf((float)deltax) : fabsf(deltax / (1.f * deltay));
    float error = 0.f;
    int y = prev.y, x = prev.x;
    const float appMag = part - 2.5f * f_log10(P.frac);
    const float bright0 = 100 * f_exp10(-.4f * appMag);
    // the reference's walk can miss (i, j) (a purely vertical move steps y
    // off the line) and then never ends; here it stops after as many steps
    // as the line is long or when it leaves the frame
    const int maxit = 2 * (abs(deltax) + abs(deltay)) + 2;
    for (int it = 0; it < maxit && (y != j || x != i); it++) {
        if (error < 1.f) {
            y += sgnDeltaY;
            error += deltaerr;
        }
        if (error >= 0.5f) {
            x += sgnDeltaX;
            error -= 1.f;
        }
        if (x < 0 || x >= H || y < 0 || y >= W) break;
        const float dist = (float)((x - i) * (x - i) + (y - j) * (y - j));
        const float fade = (traildist - sqrtf(dist)) * (traildist - sqrtf(dist)) / (traildist * traildist);
        const float brightness = bright0 * fade;
        float r, g, b;
        hsp_to_rgb(col[0], col[1], col[2] * brightness, r, g, b);
        r *= 255.f;
        g *= 255.f;
        b *= 255.f;
        const size_t ij = (size_t)x * M + y;
        trail_put(T.trail, ij, r * r, 0);
        trail_put(T.trail, ij, g * g, 1);
        trail_put(T.trail, ij, b * b, 2);
        if (dist <= 1.f) break;
    }
}

// addDiffraction (MakeImageKernel.cu:775-800): after sumStarLight the
// diffraction sprite is scattered around each pixel brighter than 255^2,
// then makePix runs.  Sources and thresholds are the light before
// diffraction (the reference reads them while other threads add to them).
// Here each output pixel gathers the contributions of the bright pixels
// whose sprite window covers it, in ascending pixel order, so the sums do
// not depend on scheduling (the reference adds with float atomics).

// Columns per entry of the bright pixels' index (a tile's width).
constexpr int kDiffCols = 16;
// Black texels around the sprite: a wave's 8 x 8 pixels reach at most seven
// beyond a window that covers one of them.
constexpr int kDiffPad = 8;

// Per frame row, the columns of its bright pixels in ascending order, their
// light over the reference's divisor 10000 * max^0.6, and how many of them lie
// left of every kDiffCols-th column (`left`, one entry more than the row has
// such groups); one wavefront per row.  Also the sprite with four bytes a
// texel, which one load reads, inside a black margin of kDiffPad texels.
__global__ __launch_bounds__(256) void diff_rows(const float* light, int W, int H, uint32_t* cols, float* scaled,
                                                 int* left, const uint8_t* sprite, int fs, uint32_t* sprite4) {
    const int pitch = fs + 2 * kDiffPad;
    for (int t = blockIdx.x * 256 + threadIdx.x; t < pitch * pitch; t += (int)gridDim.x * 256) {
        const int y = t / pitch - kDiffPad, x = t % pitch - kDiffPad;
        uint32_t v = 0;
        if (x >= 0 && x < fs && y >= 0 && y < fs) {
            const uint8_t* p = sprite + 3 * (y * fs + x);
            v = (uint32_t)p[0] | (uint32_t)p[1] << 8 | (uint32_t)p[2] << 16;
        }
        sprite4[t] = v;
    }
    const int row = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
    if (row >= H) return;
    const unsigned lane = threadIdx.x & 63;
    const int groups = (W + kDiffCols - 1) / kDiffCols;
    int* lrow = left + (size_t)row * (groups + 1);
    int n = 0;
    for (int j0 = 0; j0 < W; j0 += 64) {
        const int j = j0 + (int)lane;
        bool hot = false;
        float l0 = 0.f, l1 = 0.f, l2 = 0.f, mx = 0.f;
        if (j < W) {
            const float* l = light + 3 * ((size_t)row * W + j);
            l0 = l[0];
            l1 = l[1];
            l2 = l[2];
            mx = fmaxf(fmaxf(l0, l1), l2);
            hot = mx > 65025.f;
        }
        const unsigned long long m = __ballot(hot);
        const int at = n + __popcll(m & ((1ull << lane) - 1));
        if (lane % kDiffCols == 0 && j < W) lrow[j / kDiffCols] = at;
        if (hot) {
            const size_t o = (size_t)row * W + at;
            const float div = 10000 * f_pow(mx, 0.6f);
            cols[o] = (uint32_t)j;
            scaled[3 * o] = l0 / div;
            scaled[3 * o + 1] = l1 / div;
            scaled[3 * o + 2] = l2 / div;
        }
        n += __popcll(m);
    }
    if (lane == 0) lrow[groups] = n;
}

constexpr int kDiffCand = 512;   // bright pixels staged in LDS per round
constexpr int kDiffFly = 8;      // candidates whose sprite texels load together

// One 16 x 16 tile of output pixels per workgroup.  The bright pixels whose
// window can reach the tile are, in each row, one or (across the frame's
// edge) two runs of its list, which `left` bounds: a thread per row takes the
// runs, their lengths are summed over the rows, and the threads then fetch the
// candidates by their number, which is their pixel order.  A wave has 8 x 8
// pixels, keeps the candidates whose window reaches those, and every lane adds
// them all, kDiffFly sprite loads in flight: where the window does not cover
// its pixel it reads the sprite's black margin and adds zero (with a light
// that is no finite number, which times zero is NaN, it tests instead).  The
// window's rows outside the frame are those of no pixel.  What bounds it is
// the arithmetic of the tiles among the brightest pixels (up to 2800
// candidates a tile at 1366 x 768, 340 on average).  (One wave listing row after row, and two integer remainders per
// candidate and pixel, took 1180 us there.)
__global__ __launch_bounds__(256) void diff_gather(const float* light, const uint32_t* cols, const float* scaled,
                                                   const int* left, const uint32_t* sprite4, int fs, int W, int H,
                                                   uint8_t* img, float* o_star) {
    __shared__ float4 c_light[kDiffCand + 1];   // light, and the tile's first pixel's texel
    __shared__ short2 c_win[kDiffCand];         // that pixel's row and column of the window
    __shared__ __align__(16) uint16_t s_list[4][kDiffCand + kDiffFly];
    __shared__ int s_pre[257], s_first[256], s_len0[256], s_second[256], s_wave[4];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid / 64;
    const int wx = 8 * (wave & 1), wy = 8 * (wave / 2);
    const int tx = wx + (lane & 7), ty = wy + lane / 8;
    const int oj0 = blockIdx.x * 16, oi0 = blockIdx.y * 16;
    const int oj = oj0 + tx, oi = oi0 + ty;
    const int pitch = fs + 2 * kDiffPad;
    const unsigned texel = (unsigned)(ty * pitch + tx);
    const int fh = fs / 2;
    uint16_t* list = s_list[wave];
    if (tid == 0) c_light[kDiffCand] = make_float4(0.f, 0.f, 0.f, 0.f);   // adds nothing
    const int groups = (W + kDiffCols - 1) / kDiffCols;
    const bool mine = oi < H && oj < W;
    const size_t ij = (size_t)oi * W + oj;
    float a0 = 0.f, a1 = 0.f, a2 = 0.f;
    if (mine) {
        a0 = light[3 * ij];
        a1 = light[3 * ij + 1];
        a2 = light[3 * ij + 2];
    }
    // columns whose windows can reach the tile: c0 .. c1, c1 beyond W where they wrap
    const bool whole = 15 + fs >= W;
    int c0 = oj0 - (fs - 1 - fh);
    if (c0 < 0) c0 += W;
    const int c1 = c0 + 14 + fs;
    const bool wrap = c1 >= W;
    const int g0 = c0 / kDiffCols, g1 = (wrap ? c1 - W : c1) / kDiffCols + 1;
    // rows whose windows can reach the tile
    const int r_lo = max(0, oi0 - (fs - 1 - fh)), r_hi = min(H - 1, oi0 + 15 + fh);
    for (int rb = r_lo; rb <= r_hi; rb += 256) {
        int first = 0, len0 = 0, second = 0, len = 0;
        if (rb + tid <= r_hi) {
            const int* lrow = left + (size_t)(rb + tid) * (groups + 1);
            if (whole || (wrap && g1 >= g0)) {
                len0 = len = lrow[groups];
            } else if (wrap) {
                len0 = lrow[g1];
                second = lrow[g0];
                len = len0 + lrow[groups] - second;
            } else {
                first = lrow[g0];
                len0 = len = lrow[g1] - first;
            }
        }
        int sum = len;   // inclusive over the wave, then over the workgroup
#pragma unroll
        for (int d = 1; d < 64; d *= 2) {
            const int up = __shfl_up(sum, d);
            if (lane >= d) sum += up;
        }
        __syncthreads();   // the last batch's runs are no longer read
        if (lane == 63) s_wave[wave] = sum;
        s_first[tid] = first;
        s_len0[tid] = len0;
        s_second[tid] = second;
        __syncthreads();
        for (int w = 0; w < wave; w++) sum += s_wave[w];
        s_pre[tid + 1] = sum;
        if (tid == 0) s_pre[0] = 0;
        __syncthreads();
        const int total = s_pre[256];
        for (int x0 = 0; x0 < total; x0 += kDiffCand) {
            const int n = min(kDiffCand, total - x0);
            bool tame = true;
            for (int k = tid; k < n; k += 256) {
                const int x = x0 + k;
                int row = 0;   // the last one with s_pre[row] <= x
#pragma unroll
                for (int d = 128; d > 0; d /= 2)
                    if (s_pre[row + d] <= x) row += d;
                const int at = x - s_pre[row];
                const int r = rb + row;
                const size_t o = (size_t)r * W + (at < s_len0[row] ? s_first[row] + at : s_second[row] + at - s_len0[row]);
                const int qq = oi0 - r + fh;
                int pp = oj0 - (int)cols[o] + fh;
                if (pp < 0) pp += W;
                if (pp >= W) pp -= W;
                if (pp >= W - 15) pp -= W;   // reaches the tile from its left only
                pp = min(pp, fs);
                const float* l = scaled + 3 * o;
                c_win[k] = make_short2((short)qq, (short)pp);
                c_light[k] = make_float4(l[0], l[1], l[2], __int_as_float((qq + kDiffPad) * pitch + pp + kDiffPad));
                tame = tame && fabsf(l[0]) <= 3.4e38f && fabsf(l[1]) <= 3.4e38f && fabsf(l[2]) <= 3.4e38f;
            }
            tame = __syncthreads_and(tame);
            int m = 0;
            for (int k0 = 0; k0 < n; k0 += 64) {
                const int k = k0 + lane;
                bool reach = false;
                if (k < n) {
                    const short2 w = c_win[k];
                    reach = w.x + wy + 7 >= 0 && w.x + wy < fs && w.y + wx + 7 >= 0 && w.y + wx < fs;
                }
                const unsigned long long b = __ballot(reach);
                if (reach) list[m + __popcll(b & ((1ull << lane) - 1))] = (uint16_t)k;
                m += __popcll(b);
            }
            if (lane < kDiffFly) list[m + lane] = kDiffCand;
            __builtin_amdgcn_wave_barrier();
            const auto add = [&](const float4& l, uint32_t px) {
                const float dx = l.x * (float)(px & 255u), dy = l.y * (float)(px >> 8 & 255u),
                            dz = l.z * (float)(px >> 16 & 255u);
                a0 += fminf(65025.f, dx * dx);
                a1 += fminf(65025.f, dy * dy);
                a2 += fminf(65025.f, dz * dz);
            };
            if (tame) {
                for (int k = 0; k < m; k += kDiffFly) {
                    uint32_t px[kDiffFly];
                    float4 l[kDiffFly];
#pragma unroll
                    for (int u = 0; u < kDiffFly; u++) {
                        l[u] = c_light[list[k + u]];
                        px[u] = sprite4[(unsigned)__float_as_int(l[u].w) + texel];
                    }
#pragma unroll
                    for (int u = 0; u < kDiffFly; u++) add(l[u], px[u]);
                }
            } else {
                for (int k = 0; k < m; k++) {
                    const short2 w = c_win[list[k]];
                    const float4 l = c_light[list[k]];
                    if ((unsigned)(w.x + ty) < (unsigned)fs && (unsigned)(w.y + tx) < (unsigned)fs)
                        add(l, sprite4[(unsigned)__float_as_int(l.w) + texel]);
                }
            }
            __syncthreads();
        }
    }
    if (!mine) return;
    make_pix(a0, a1, a2, img, ij);
    if (o_star) {
        o_star[3 * ij] = a0;
        o_star[3 * ij + 1] = a1;
        o_star[3 * ij + 2] = a2;
    }
}

// ---- distortEnvironmentMap (MakeImageKernel.cu:631-751) ----
// A pixel sums one summed-table difference per sky column of its footprint,
// in column order.  env_map does pixels of at most kInlineCols columns (95%
// of a lensed 1080p frame), one lane each; env_map_group those of up to
// kGroupCols, sixteen lanes each; env_map_heavy the rest, one wavefront each.
// The first line: env_map + env_map_group took 241, 178, 157, 149 and 174 us
// of a 1080p frame, and 576, 373, 354, 344 and 368 us of a 4K one, with
// kInlineCols 8, 32, 48, 64 and 96 (and 45, 51, 59, 61, 80 us at 320x180,
// beside a longer star pass): a lane keeps eight loads in flight and
// finishes its own pixel, a group of sixteen pays its scan and its staging.

constexpr int kInlineCols = 64;
constexpr int kGroupCols = 256;

struct EnvPix {
    float t[4], p[4];
    float slope[4];   // of edge q, theta over phi
    int ind, pixMin, pixNum;
    float thMax, thMin;
};

// The sky: summed table, its size, the size of a texel and the inverse of
// that in FP64.
struct SkyK {
    const float4* table;
    int rows, cols;
    float pixSize;
    double inv;
};

// Texel index of an angle: cvt_i32(x / pixSize).  The FP64 product with the
// rounded inverse is within 2^-52 of the quotient, and a quotient of two
// 24-bit numbers is no 25-bit one and at least 2^-49 from any, so it rounds
// to the same float as the division (a third of its instructions).
__device__ __forceinline__ int texel(const SkyK& K, float x) { return cvt_i32((float)((double)x * K.inv)); }

// Corners and column range of pixel (i, j); false for pixel index 0 (the
// reference's `ind > 0`, MakeImageKernel.cu:647), which stays black.
__device__ __forceinline__ bool env_setup(const float* thphi, int W, int i, int j, float offset, const SkyK& K,
                                          EnvPix& E) {
    bool picheck = false;
    E.ind = i * (W + 1) + j;
    corners(thphi, W, E.ind, E.t, E.p, picheck, offset);
    if (E.ind <= 0) return false;
    float phMax = fmaxf(fmaxf(E.p[0], E.p[1]), fmaxf(E.p[2], E.p[3]));
    float phMin = fminf(fminf(E.p[0], E.p[1]), fminf(E.p[2], E.p[3]));
    int pixMax = texel(K, phMax);
    E.pixMin = texel(K, phMin);
    E.pixNum = pixMax - E.pixMin + 1;
    if (E.pixNum > 1 && pixMax * K.pixSize > phMax) E.pixNum -= 1;
    E.thMax = fmaxf(fmaxf(E.t[0], E.t[1]), fmaxf(E.t[2], E.t[3]));
    E.thMin = fminf(fminf(E.t[0], E.t[1]), fminf(E.t[2], E.t[3]));
    return true;
}

__device__ __forceinline__ void env_slopes(EnvPix& E) {
#pragma unroll
    for (int q = 0; q < 4; q++)
        E.slope[q] = (E.t[(q + 1) % 4] - E.t[q]) / (E.p[(q + 1) % 4] - E.p[q]);
}

// The quad's theta span on the column boundary at phi = cp, folded into the
// running (mn, mx) (the reference never resets it between boundaries).
__device__ __forceinline__ void env_boundary(const EnvPix& E, float cp, float& mn, float& mx) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
        float ap = E.p[q], bp = E.p[(q + 1) % 4];
        float ct = E.t[q] + E.slope[q] * (cp - ap);
        const bool on = (cp - ap) * (cp - bp) <= 0;
        mn = on && ct < mn ? ct : mn;
        mx = on && ct > mx ? ct : mx;
    }
}

// Table indices of the two ends of column `col` over the running span; lo < 0: no lower end.
__device__ __forceinline__ void env_ends(const SkyK& K, int col, float mn, float mx, int& hi, int& lo) {
    hi = min(max(texel(K, mx), 0), K.rows - 1) * K.cols + col;
    const int index2 = (texel(K, mn) - 1) * K.cols + col;
    lo = index2 <= 0 ? -1 : index2 >= K.rows * K.cols ? (K.rows - 1) * K.cols + col : index2;
}

__device__ __forceinline__ float4 env_diff(float4 mxc, float4 mnc) {
    return make_float4(mxc.x - mnc.x, mxc.y - mnc.y, mxc.z - mnc.z, mxc.w - mnc.w);
}

// Summed-table difference of column `col` over the running span.
__device__ __forceinline__ float4 env_column(const SkyK& K, int col, float mn, float mx) {
    int hi, lo;
    env_ends(K, col, mn, mx, hi, lo);
    const float4 mxc = K.table[hi];
    float4 mnc = make_float4(0.f, 0.f, 0.f, 0.f);
    if (lo >= 0) mnc = K.table[lo];
    return env_diff(mxc, mnc);
}

// Mean colour -> gamma -> HSP -> lensing/redshift -> BGRA (MakeImageKernel.cu:733-750).
__device__ __forceinline__ uchar4 env_finish(const EnvPix& E, float cx, float cy, float cz, float cw, int W,
                                             int lr, const Cam7& cam, const float* view, float area_ij) {
    // FP32 pow of the device library (a few ulps, as the reference's own
    // powf): these values only reach the 8-bit output
    cx = fminf(255.f, powf(cx / cw, 1.f / 2.2f));
    cy = fminf(255.f, powf(cy / cw, 1.f / 2.2f));
    cz = fminf(255.f, powf(cz / cw, 1.f / 2.2f));
    float Hh, Ss, Pp;
    rgb_to_hsp(cz / 255.f, cy / 255.f, cx / 255.f, Hh, Ss, Pp);
    if (lr) {
        float redshft, frac;
        lensing_redshift(E.t, E.p, W, E.ind, cam, view, frac, redshft, area_ij);
        Pp *= frac;
        Pp = powf(Pp, redshft);
    }
    hsp_to_rgb(Hh, Ss, fminf(1.f, Pp), cz, cy, cx);
    uchar4 o;
    o.x = (uint8_t)min(255, cvt_i32(cx * 255));
    o.y = (uint8_t)min(255, cvt_i32(cy * 255));
    o.z = (uint8_t)min(255, cvt_i32(cz * 255));
    o.w = 255;
    return o;
}

// Column sums of a pixel in the reference's order (one lane).
__device__ __forceinline__ float4 env_seq(EnvPix& E, const SkyK& K) {
    const int cols = K.cols;
    float cx = 0.f, cy = 0.f, cz = 0.f, cw = 0.f;
    if (E.pixNum == 1) {
        int rmax = min(max(texel(K, E.thMax), 0), K.rows - 1);
        int rmin = texel(K, E.thMin) - 1;
        int col = min(max(E.pixMin, 0), cols - 1);
        float4 mxc = K.table[(size_t)rmax * cols + col];
        float4 mnc = make_float4(0.f, 0.f, 0.f, 0.f);
        if (rmin >= 0) mnc = K.table[(size_t)min(rmin, K.rows - 1) * cols + col];
        cx = mxc.x - mnc.x;
        cy = mxc.y - mnc.y;
        cz = mxc.z - mnc.z;
        cw = mxc.w - mnc.w;
    } else if (E.pixNum < cols) {
        env_slopes(E);
        float mx = -100, mn = cols + 1;
        env_boundary(E, E.pixMin * K.pixSize, mn, mx);
        int col = E.pixMin % cols;
        // four columns at a time: their loads are in flight together, their
        // terms are added in column order
        for (int s0 = 1; s0 <= E.pixNum; s0 += 4) {
            float4 a[4], b[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                a[u] = b[u] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (s0 + u <= E.pixNum) {
                    env_boundary(E, (E.pixMin + s0 + u) * K.pixSize, mn, mx);
                    col = col + 1 == cols ? 0 : col + 1;
                    int hi, lo;
                    env_ends(K, col, mn, mx, hi, lo);
                    a[u] = K.table[hi];
                    if (lo >= 0) b[u] = K.table[lo];
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (s0 + u <= E.pixNum) {
                    const float4 d = env_diff(a[u], b[u]);
                    cx += d.x;
                    cy += d.y;
                    cz += d.z;
                    cw += d.w;
                }
        }
    } else {
        int thMaxPix = min(max(texel(K, E.thMax), 0), K.rows - 1) * cols;
        int thMinPix = min(max(texel(K, E.thMin), 0), K.rows - 1) * cols;
        for (int q = 0; q < E.pixNum; q++) {
            float4 mxc = K.table[thMaxPix + (E.pixMin + q) % cols];
            float4 mnc = K.table[thMinPix + (E.pixMin + q) % cols];
            cx += mxc.x - mnc.x;
            cy += mxc.y - mnc.y;
            cz += mxc.z - mnc.z;
            cw += mxc.w - mnc.w;
        }
    }
    return make_float4(cx, cy, cz, cw);
}

// env counters, each on a line of its own: entries of the group and the heavy queue
constexpr int kCtrGroup = 0, kCtrHeavy = 32, kEnvCtrWords = 64;

__global__ __launch_bounds__(256) void env_map(const float* thphi, const uint8_t* bh, SkyK K, Cam7 cam, int W,
                                               int H, float offset, int lr, const float* area,
                                               const float* view, uint8_t* img, uint32_t* qgroup, uint32_t* qwave,
                                               unsigned* nq) {
    __shared__ uint32_t s_q[2][256];
    __shared__ unsigned s_n[2], s_base[2];
    const unsigned tid = threadIdx.y * 16 + threadIdx.x;
    if (tid < 2) s_n[tid] = 0;
    __syncthreads();
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    const bool valid = i < H && j < W;
    const size_t ij = valid ? (size_t)i * W + j : 0;
    EnvPix E;
    const bool live = valid && bh[ij] == 0 && env_setup(thphi, W, i, j, offset, K, E);
    const int tier = !live || E.pixNum <= kInlineCols ? 0 : E.pixNum <= kGroupCols ? 1 : 2;
    if (tier) s_q[tier - 1][atomicAdd(&s_n[tier - 1], 1u)] = (uint32_t)ij;
    __syncthreads();
    // one append per workgroup and queue
    if (tid < 2 && s_n[tid]) s_base[tid] = atomicAdd(&nq[tid ? kCtrHeavy : kCtrGroup], s_n[tid]);
    __syncthreads();
    if (tid < s_n[0]) qgroup[s_base[0] + tid] = s_q[0][tid];
    if (tid < s_n[1]) qwave[s_base[1] + tid] = s_q[1][tid];
    if (!valid || tier != 0) return;   // env_map_group / env_map_heavy write this pixel
    uchar4 o = make_uchar4(0, 0, 0, 255);
    if (live) {
        float4 c4 = env_seq(E, K);
        o = env_finish(E, c4.x, c4.y, c4.z, c4.w, W, lr, cam, view, area[ij]);
    }
    reinterpret_cast<uchar4*>(img)[ij] = o;
}

// The block's place in an order in which the blocks of one XCD (blocks go to
// the eight XCDs in turn) are neighbours: neighbouring pixels of a queue read
// the same sky rows, and then find them in their XCD's L2.  The grid is a
// multiple of 8 blocks.
__device__ __forceinline__ unsigned xcd_block() { return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

// Sixteen lanes per queued pixel: a lane takes every sixteenth column
// boundary, the running span (an exact min/max) is scanned over the lanes,
// the sixteen columns' loads are in flight together, and their terms, staged
// in LDS, are added in column order, one colour component per lane.  A wave
// takes 64 pixels (fewer where the queue does not fill the launch) and
// finishes their means together.  (One lane per pixel, column after column,
// took 180 us of every frame, however small.)
constexpr int kGroupLanes = 16, kGroupPix = 64 / kGroupLanes;   // a 16-lane DPP row per pixel

// One step of the inclusive min/max scan over a 16-lane row: CTRL is the DPP
// row shift; lanes shifted in from outside the row keep their own values.
template <int CTRL>
__device__ __forceinline__ void row_scan(float& mn, float& mx) {
    const float a = __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(mn), __float_as_int(mn), CTRL, 0xf, 0xf, false));
    const float b = __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(mx), __float_as_int(mx), CTRL, 0xf, 0xf, false));
    mn = fminf(mn, a);
    mx = fmaxf(mx, b);
}

__global__ __launch_bounds__(256) void env_map_group(const float* thphi, SkyK K, Cam7 cam, int W, float offset,
                                                     int lr, const float* area, const float* view, uint8_t* img,
                                                     const uint32_t* queue, const unsigned* nq) {
    __shared__ float4 s_d[4][64];     // per wave: the terms of kGroupPix pixels x kGroupLanes columns
    __shared__ float s_c[4][64][4];   // per wave: the sums of its pixels
    const unsigned n = *nq;
    const unsigned lane = threadIdx.x & 63, wslot = threadIdx.x >> 6;
    const unsigned sub = lane % kGroupLanes, grp = lane / kGroupLanes;
    const unsigned nwaves = gridDim.x * 4;
    const unsigned rounds = min(64u / kGroupPix, max(1u, n / (kGroupPix * nwaves)));
    const unsigned per = rounds * kGroupPix;   // pixels a wave takes at a time
    const int cols = K.cols;
    for (unsigned e0 = (xcd_block() * 4 + wslot) * per; e0 < n; e0 += nwaves * per) {
        for (unsigned r = 0; r < rounds; r++) {
            const unsigned e = e0 + r * kGroupPix + grp;
            int num = -1;   // last boundary; -1: nothing to do here
            EnvPix E;
            if (e < n) {
                const uint32_t ij = queue[e];
                env_setup(thphi, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, K, E);
                env_slopes(E);
                if (E.pixNum < cols) num = E.pixNum;
            }
            float sum = 0.f, cmn = cols + 1, cmx = -100;   // (cmn, cmx): the span after the columns so far
            int col = num >= 0 ? (E.pixMin + (int)sub) % cols : 0;
            for (int s0 = 0; __ballot(s0 <= num); s0 += kGroupLanes) {
                const int sidx = s0 + (int)sub;
                float mn = cols + 1, mx = -100;
                if (sidx <= num) env_boundary(E, (E.pixMin + sidx) * K.pixSize, mn, mx);
                row_scan<0x111>(mn, mx);
                row_scan<0x112>(mn, mx);
                row_scan<0x114>(mn, mx);
                row_scan<0x118>(mn, mx);
                mn = fminf(mn, cmn);
                mx = fmaxf(mx, cmx);
                cmn = __shfl(mn, kGroupLanes - 1, kGroupLanes);
                cmx = __shfl(mx, kGroupLanes - 1, kGroupLanes);
                float4 d = make_float4(0.f, 0.f, 0.f, 0.f);
                if (sidx > 0 && sidx <= num) d = env_column(K, col, mn, mx);
                col += kGroupLanes;
                while (col >= cols) col -= cols;
                __builtin_amdgcn_wave_barrier();
                s_d[wslot][lane] = d;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (sub < 4) {
                    const float* x = reinterpret_cast<const float*>(&s_d[wslot][grp * kGroupLanes]) + sub;
                    float v[kGroupLanes];
#pragma unroll
                    for (int u = 0; u < kGroupLanes; u++) v[u] = x[4 * u];
#pragma unroll
                    for (int u = 0; u < kGroupLanes; u++) sum += v[u];   // a term outside the footprint is zero
                }
            }
            if (sub < 4) s_c[wslot][r * kGroupPix + grp][sub] = sum;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane < per && e0 + lane < n) {
            const uint32_t ij = queue[e0 + lane];
            EnvPix E;
            env_setup(thphi, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, K, E);
            const float* c = s_c[wslot][lane];
            float4 c4 = make_float4(c[0], c[1], c[2], c[3]);
            if (E.pixNum >= cols) c4 = env_seq(E, K);   // a sky of fewer columns than the footprint's
            reinterpret_cast<uchar4*>(img)[ij] = env_finish(E, c4.x, c4.y, c4.z, c4.w, W, lr, cam, view, area[ij]);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

__device__ __forceinline__ float read_lane(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__device__ __forceinline__ float wave_xor_sum(float v) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v += __shfl_xor(v, off);
    return v;
}

// One wavefront per queued pixel.  The sum's order: the column boundaries are
// cut into 64 contiguous chunks, each chunk's terms are added in order, and
// the 64 sums by an xor butterfly.  The terms are made 64 neighbouring
// columns at a time, one per lane (the running theta span is an exact
// min/max, scanned over the lanes), so that the table is read in whole
// lines, and staged in LDS, kHeavyWindow of them; then the lanes add the
// terms of their chunks.  (A lane walking its own chunk through memory read
// every line about twice and made every boundary twice: 277 us of a 1080p
// frame's sky pass.)  A wave finishes the means of its pixels together, one
// per lane.
constexpr int kHeavyWindow = 512;

__global__ __launch_bounds__(128) void env_map_heavy(const float* thphi, SkyK K, Cam7 cam, int W,
                                                     float offset, int lr, const float* area, const float* view,
                                                     uint8_t* img, const uint32_t* heavy, const unsigned* nheavy) {
    __shared__ float4 s_c[2][64];
    __shared__ float4 s_d[2][kHeavyWindow];
    const unsigned lane = threadIdx.x & 63, wslot = threadIdx.x >> 6;
    const unsigned wave = xcd_block() * 2 + wslot;
    const unsigned nwaves = gridDim.x * 2;
    const unsigned n = *nheavy;
    const int rows = K.rows, cols = K.cols;
    // pixel wave + k nwaves is the wave's k-th
    for (unsigned e0 = wave; e0 < n; e0 += 64 * nwaves) {
        unsigned cnt = 0;
        for (; cnt < 64 && e0 + cnt * nwaves < n; cnt++) {
            const uint32_t ij = heavy[e0 + cnt * nwaves];
            EnvPix E;
            env_setup(thphi, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, K, E);
            float cx = 0.f, cy = 0.f, cz = 0.f, cw = 0.f;
            if (E.pixNum < cols) {
                env_slopes(E);
                const int nb = E.pixNum + 1;   // boundaries 0..pixNum
                const int per = (nb + 63) / 64;
                int next = min((int)lane * per, nb);   // the chunk's next term
                const int end = min(next + per, nb);
                float cmn = cols + 1, cmx = -100;      // the span after the boundaries so far
                int col = (E.pixMin + (int)lane) % cols;
                for (int w0 = 0; w0 < nb; w0 += kHeavyWindow) {
                    for (int b4 = 0; b4 < kHeavyWindow && w0 + b4 < nb; b4 += 256) {
                      int ihi[4], ilo[4];
#pragma unroll
                      for (int u = 0; u < 4; u++) {
                        const int b = w0 + b4 + 64 * u + (int)lane;
                        float mn = cols + 1, mx = -100;
                        if (b < nb) env_boundary(E, (E.pixMin + b) * K.pixSize, mn, mx);
                        // inclusive scan over the rows of 16, then over the rows
                        row_scan<0x111>(mn, mx);
                        row_scan<0x112>(mn, mx);
                        row_scan<0x114>(mn, mx);
                        row_scan<0x118>(mn, mx);
                        const float n0 = read_lane(mn, 15), n1 = read_lane(mn, 31), n2 = read_lane(mn, 47),
                                    n3 = read_lane(mn, 63);
                        const float x0 = read_lane(mx, 15), x1 = read_lane(mx, 31), x2 = read_lane(mx, 47),
                                    x3 = read_lane(mx, 63);
                        const float n01 = fminf(n0, n1), x01 = fmaxf(x0, x1);
                        const float n02 = fminf(n01, n2), x02 = fmaxf(x01, x2);
                        const unsigned row = lane >> 4;
                        mn = fminf(fminf(mn, cmn), row == 0 ? mn : row == 1 ? n0 : row == 2 ? n01 : n02);
                        mx = fmaxf(fmaxf(mx, cmx), row == 0 ? mx : row == 1 ? x0 : row == 2 ? x01 : x02);
                        cmn = fminf(cmn, fminf(n02, n3));
                        cmx = fmaxf(cmx, fmaxf(x02, x3));
                        ihi[u] = ilo[u] = -1;
                        if (b > 0 && b < nb) env_ends(K, col, mn, mx, ihi[u], ilo[u]);
                        col += 64;
                        while (col >= cols) col -= cols;
                      }
                      float4 x[4], y[4];
#pragma unroll
                      for (int u = 0; u < 4; u++) {
                        x[u] = y[u] = make_float4(0.f, 0.f, 0.f, 0.f);
                        if (ihi[u] >= 0) x[u] = K.table[ihi[u]];
                        if (ilo[u] >= 0) y[u] = K.table[ilo[u]];
                      }
#pragma unroll
                      for (int u = 0; u < 4; u++) s_d[wslot][b4 + 64 * u + lane] = env_diff(x[u], y[u]);
                    }
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    const int stop = min(end, w0 + kHeavyWindow);
                    for (; next < stop; next++) {
                        const float4 d = s_d[wslot][next - w0];   // term 0 is zero
                        cx += d.x;
                        cy += d.y;
                        cz += d.z;
                        cw += d.w;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                }
            } else {
                int thMaxPix = min(max(texel(K, E.thMax), 0), rows - 1) * cols;
                int thMinPix = min(max(texel(K, E.thMin), 0), rows - 1) * cols;
                for (int q = lane; q < E.pixNum; q += 64) {
                    float4 mxc = K.table[thMaxPix + (E.pixMin + q) % cols];
                    float4 mnc = K.table[thMinPix + (E.pixMin + q) % cols];
                    cx += mxc.x - mnc.x;
                    cy += mxc.y - mnc.y;
                    cz += mxc.z - mnc.z;
                    cw += mxc.w - mnc.w;
                }
            }
            cx = wave_xor_sum(cx);
            cy = wave_xor_sum(cy);
            cz = wave_xor_sum(cz);
            cw = wave_xor_sum(cw);
            if (lane == 0) s_c[wslot][cnt] = make_float4(cx, cy, cz, cw);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane < cnt) {
            const uint32_t ij = heavy[e0 + lane * nwaves];
            EnvPix E;
            env_setup(thphi, W, (int)(ij / (uint32_t)W), (int)(ij % (uint32_t)W), offset, K, E);
            const float4 c4 = s_c[wslot][lane];
            reinterpret_cast<uchar4*>(img)[ij] = env_finish(E, c4.x, c4.y, c4.z, c4.w, W, lr, cam, view, area[ij]);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// addStarsAndBackground (MakeImageKernel.cu:837-853)
__global__ __launch_bounds__(256) void composite(const uint8_t* img_star, const uint8_t* img_map, int64_t n,
                                                 int star, int map, uint8_t* out) {
    int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    uchar4 o;
    if (star && map) {
        uchar4 s = reinterpret_cast<const uchar4*>(img_star)[q];
        uchar4 b = reinterpret_cast<const uchar4*>(img_map)[q];
        float p = 1.f;
        float sx = (float)s.x * s.x, sy = (float)s.y * s.y, sz = (float)s.z * s.z;
        float bx = (float)b.x * b.x, by = (float)b.y * b.y, bz = (float)b.z * b.z;
        o.x = (uint8_t)min(cvt_i32(sqrtf(p * sx + (2.f - p) * bx)), 255);
        o.y = (uint8_t)min(cvt_i32(sqrtf(p * sy + (2.f - p) * by)), 255);
        o.z = (uint8_t)min(cvt_i32(sqrtf(p * sz + (2.f - p) * bz)), 255);
        o.w = 255;
    } else if (map) {
        o = reinterpret_cast<const uchar4*>(img_map)[q];
    } else if (star) {
        o = reinterpret_cast<const uchar4*>(img_star)[q];
    } else {
        o = make_uchar4(0, 0, 0, 255);
    }
    reinterpret_cast<uchar4*>(out)[q] = o;
}

// Summed-area sky table (MakeImageKernel.cu:1312-1331) in two passes: the
// terms of every texel, then their sums down the columns in the reference's
// order.  (One thread per column doing both had 64 waves, each a chain of
// `rows` texels of eight trigonometric functions and three pows: 5.86 ms of a
// 4096 x 2048 sky.)
//
// Terms: colour^2.2 * solid angle per channel, and the solid angle.  A texel's
// corners lie on the lattice pxsz * k in both angles, so a block of
// kSumCols x kSumRows texels needs the sines and cosines of its lattice lines
// only, and a channel value has 256 powers: both are taken once per block and
// read from LDS, and the texel keeps its two arctangents.
constexpr int kSumCols = 64, kSumRows = 32;

__global__ __launch_bounds__(256) void sum_terms(const uint8_t* sky, int rows, int cols, float* table) {
    __shared__ float s_pow[256];
    __shared__ float s_st[kSumRows + 1], s_ct[kSumRows + 1], s_sp[kSumCols + 1], s_cp[kSumCols + 1];
    const float pxsz = BT_FPI2 / (1.f * cols);
    const int q0 = blockIdx.x * kSumCols, p0 = blockIdx.y * kSumRows;
    const int tid = threadIdx.x;
    s_pow[tid] = f_pow((float)tid, 2.2f);
    if (tid <= kSumCols) {
        const float phi = pxsz * (q0 + tid);
        s_sp[tid] = f_sin(phi);
        s_cp[tid] = f_cos(phi);
    } else if (tid >= 128 && tid <= 128 + kSumRows) {
        const float theta = pxsz * (p0 + tid - 128);
        s_st[tid - 128] = f_sin(theta);
        s_ct[tid - 128] = f_cos(theta);
    }
    __syncthreads();
    const int dq = tid % kSumCols, q = q0 + dq;
    if (q >= cols) return;
    for (int dp = tid / kSumCols; dp < kSumRows && p0 + dp < rows; dp += 256 / kSumCols) {
        // corners: (theta below, phi), (above, phi), (above, phi + 1), (below, phi + 1)
        const float sb = s_st[dp + 1], sa = s_st[dp];
        const float x[4] = {sb * s_cp[dq], sa * s_cp[dq], sa * s_cp[dq + 1], sb * s_cp[dq + 1]};
        const float y[4] = {sb * s_sp[dq], sa * s_sp[dq], sa * s_sp[dq + 1], sb * s_sp[dq + 1]};
        const float z[4] = {s_ct[dp + 1], s_ct[dp], s_ct[dp], s_ct[dp + 1]};
        const float area = area4_of(x, y, z);
        const size_t o = (size_t)(p0 + dp) * cols + q;
        const uint8_t* px = sky + 3 * o;
        reinterpret_cast<float4*>(table)[o] =
            make_float4(s_pow[px[0]] * area, s_pow[px[1]] * area, s_pow[px[2]] * area, area);
    }
}

// Sums down the columns, in place: one lane per column and component, so a
// wave's row is one 256-byte line, and a row's four sums do not share a lane.
// The chain is one addition a row; what bounds it is the memory round trip,
// so the next kSumAhead rows are in flight while this batch is added.
constexpr int kSumAhead = 16;

__global__ __launch_bounds__(64) void sum_columns(int rows, size_t stride, float* table) {
    const size_t g = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (g >= stride) return;
    float* t = table + g;
    float sum = 0.f, next[kSumAhead];
#pragma unroll
    for (int k = 0; k < kSumAhead; k++) next[k] = k < rows ? t[k * stride] : 0.f;
    for (int p = 0; p < rows; p += kSumAhead) {
        float cur[kSumAhead];
#pragma unroll
        for (int k = 0; k < kSumAhead; k++) cur[k] = next[k];
#pragma unroll
        for (int k = 0; k < kSumAhead; k++) {
            const int r = p + kSumAhead + k;
            if (r < rows) next[k] = t[r * stride];
        }
#pragma unroll
        for (int k = 0; k < kSumAhead; k++) {
            if (p + k >= rows) break;
            sum += cur[k];
            t[(p + k) * stride] = sum;
        }
    }
}

// makeGrid (MakeImageKernel.cu:369-384) with hashLookup (kernel.cuh:705-733), G == 1.
__global__ void make_grid(const float* ht, const int32_t* ot, const int32_t* tag, int hw, int ow, int GN, int GM,
                          int sym, int GN1, float* grid) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= GN || j >= GM) return;
    int ix = (i + ow) % ow, iy = (j + ow) % ow;
    int ax = (i + hw) % hw + ot[2 * (ix * ow + iy)];
    int ay = (j + hw) % hw + ot[2 * (ix * ow + iy) + 1];
    int hx = (ax + hw) % hw, hy = (ay + hw) % hw;
    int sidx = hx * hw + hy;
    float vx = -2.f, vy = -2.f;
    if (tag[2 * sidx] == i && tag[2 * sidx + 1] == j) {
        vx = ht[2 * sidx];
        vy = ht[2 * sidx + 1];
    }
    float2* g2 = reinterpret_cast<float2*>(grid);
    g2[(size_t)i * GM + j] = make_float2(vx, vy);
    if (sym == 1) {
        if (vx != -1 && vx != -2) vx = BT_FPI - vx;
        int x = GN1 - i - 1;
        g2[(size_t)x * GM + j] = make_float2(vx, vy);
    }
}

// Dense FP32 grid from a device-built FP64 grid: the values saveAsGpuHash
// would store (Grid.h:645-650), without the hash round trip.
__global__ void grid_to_f32(const double* cel, int GN, int GM, int sym, int GN1, float* grid) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int i = blockIdx.y * blockDim.y + threadIdx.y;
    if (i >= GN || j >= GM) return;
    size_t o = (size_t)i * GM + j;
    float vx = (float)cel[2 * o], vy = (float)cel[2 * o + 1];
    float2* g2 = reinterpret_cast<float2*>(grid);
    g2[o] = make_float2(vx, vy);
    if (sym == 1) {
        if (vx != -1 && vx != -2) vx = BT_FPI - vx;
        int x = GN1 - i - 1;
        g2[(size_t)x * GM + j] = make_float2(vx, vy);
    }
}

GridV grid_view(const GridF& g) {
    return GridV{g.grid, g.GN, g.GM, (g.GM & (g.GM - 1)) == 0 ? 1.f / (float)g.GM : 0.f};
}

int few_span(size_t NP) {
    int span = 256;
    while (span < kFewSpan && (size_t)span * 1024 < NP) span *= 2;
    return span;
}

// The pixels that one lane each traces: those of few candidates, then the
// odd ones among them.
template <int STEP>
void star_rest(Context* c, hipStream_t st, const float* thphi, const uint8_t* bh, const SceneK& s,
               const Cam7& cam, int W, int H, const bt_render_flags& f, const float* area, const float* view,
               float* taps, const StarQueue& Q) {
    KTimer t(c, "star_odd", st);
    const size_t NP = (size_t)W * H;
    const int span = few_span(NP);
    star_few<STEP><<<(unsigned)((NP + span - 1) / span), 256, 0, st>>>(thphi, bh, s, cam, W, H, f.offset, f.lr, area,
                                                                       view, taps, Q, span);
    star_map_odd<STEP><<<(unsigned)c->num_cus, 256, 0, st>>>(thphi, bh, s, cam, W, H, f.offset, f.lr, area, view, taps,
                                                             Q);
}

dim3 grid2d(int W, int H) { return dim3((unsigned)((W + 15) / 16), (unsigned)((H + 15) / 16)); }

}  // namespace

int render_sum_table(Context* c, const uint8_t* d_sky, int rows, int cols, float* d_table) {
    KTimer t(c, "sum_table");
    const dim3 blocks((unsigned)((cols + kSumCols - 1) / kSumCols), (unsigned)((rows + kSumRows - 1) / kSumRows));
    sum_terms<<<blocks, 256, 0, c->stream>>>(d_sky, rows, cols, d_table);
    const size_t stride = 4 * (size_t)cols;
    sum_columns<<<(unsigned)((stride + 63) / 64), 64, 0, c->stream>>>(rows, stride, d_table);
    BT_HIP(hipGetLastError());
    return BT_OK;
}

int render_grid_from_psh(Context* c, const float* d_ht, const int32_t* d_ot, const int32_t* d_tag, int hw,
                         int ow, int GN, int GM, float* d_grid, int* GN1_out) {
    int sym = (float)GM / (float)GN > 3 ? 1 : 0;
    int GN1 = sym ? 2 * GN - 1 : GN;
    KTimer t(c, "make_grid");
    make_grid<<<grid2d(GM, GN), dim3(16, 16), 0, c->stream>>>(d_ht, d_ot, d_tag, hw, ow, GN, GM, sym, GN1, d_grid);
    BT_HIP(hipGetLastError());
    *GN1_out = GN1;
    return BT_OK;
}

int render_grid_from_cel(Context* c, const double* d_cel, int GN, int GM, float* d_grid, int* GN1_out) {
    int sym = (float)GM / (float)GN > 3 ? 1 : 0;
    int GN1 = sym ? 2 * GN - 1 : GN;
    KTimer t(c, "grid_to_f32");
    grid_to_f32<<<grid2d(GM, GN), dim3(16, 16), 0, c->stream>>>(d_cel, GN, GM, sym, GN1, d_grid);
    BT_HIP(hipGetLastError());
    *GN1_out = GN1;
    return BT_OK;
}

int view_pixel_areas(Context* c, const float* view, int W, int H, float* out) {
    view_pixel_areas<<<grid2d(W, H), dim3(16, 16), 0, c->stream>>>(view, W, H, out);
    BT_HIP(hipGetLastError());
    return BT_OK;
}

size_t frame_bytes(int w, int h, int step) {
    const size_t NP = (size_t)w * h, NC = (size_t)(w + 1) * (h + 1);
    const size_t fw = 2 * (size_t)step + 1;
    // thphi, gap | bh, area x2, star and map images, per-tap star light,
    // star chunk partials, star queues (6), odd pixels and lensing (3), env queues (2),
    // lit-pixel flags, tree ranges (NP / 4 + 65536 of 8 B), BGRA output
    return NC * (8 + 4) + NP * (1 + 4 + 4 + 4 + 4 + 12 * fw * fw + 12 * fw * fw + 28 + 12 + 8 + 2 + 4 + 1) + 4096 +
           65536 * 8;
}

int render_frame(Context* c, const GridF& g, const SceneK& s, const ViewK& v, const float* cam7,
                 const bt_render_flags& f, int step, uint8_t* d_out, FrameDebug* dbg, const Blend* blend,
                 const TrailFrame* tf) {
    const int W = v.W, H = v.H;
    const size_t NP = (size_t)W * H, NC = (size_t)(W + 1) * (H + 1);
    if (step != 1 && step != 2 && step != 3)
        return fail(BT_ERR_INVALID, "render: star splat step must be 1, 2 or 3");
    // the reference's frame offset is 2*pi*q/(...) >= 0 (MakeImageKernel.cu:1413); the sky
    // lookups assume phi + offset >= 0
    if (!(f.offset >= 0.f) || !std::isfinite(f.offset) || !std::isfinite(f.hor) || !std::isfinite(f.ver))
        return fail(BT_ERR_INVALID, "render: offset must be finite and >= 0; hor/ver finite");
    if (W <= 0 || H <= 0 || g.GN < 2 || g.GM < 2 || s.rows <= 0 || s.cols <= 0)
        return fail(BT_ERR_INVALID, "render: empty frame, grid or sky");
    if (tf && (tf->W != W || tf->H != H))
        return fail(BT_ERR_INVALID, "render: the trail state was made for another frame size");
    if (tf && tf->k.S != s.S) return fail(BT_ERR_INVALID, "render: the trail state was made for another star set");
    if (blend && (blend->b.GN != g.GN || blend->b.GM != g.GM || blend->b.gridlvl != g.gridlvl || !blend->border ||
                  !(blend->alpha >= 0.f && blend->alpha <= 1.f)))
        return fail(BT_ERR_INVALID, "render: blended grids must have equal sizes and levels; alpha in [0, 1]");
    void* p;
    int rc;
    if ((rc = c->buffer("r_thphi", sizeof(float) * 2 * NC, &p))) return rc;
    float* thphi = (float*)p;
    if ((rc = c->buffer("r_gap", sizeof(int) * NC, &p))) return rc;
    int* gap = (int*)p;
    if ((rc = c->buffer("r_bh", NP, &p))) return rc;
    uint8_t* bh = (uint8_t*)p;
    if ((rc = c->buffer("r_area", sizeof(float) * NP, &p))) return rc;
    float* area = (float*)p;
    if ((rc = c->buffer("r_area_s", sizeof(float) * (NP + 64), &p))) return rc;
    float* area_s = (float*)p;
    if ((rc = c->buffer("r_img_star", 4 * NP, &p))) return rc;
    uint8_t* img_star = (uint8_t*)p;
    if ((rc = c->buffer("r_img_map", 4 * NP, &p))) return rc;
    uint8_t* img_map = (uint8_t*)p;

    // the counters of the star and the sky queues, cleared by bh_area
    if ((rc = c->buffer("r_queue_ctr", sizeof(unsigned) * (kStarCtrWords + kEnvCtrWords), &p))) return rc;
    unsigned* ctr = (unsigned*)p;

    Cam7 cam;
    for (int q = 0; q < 7; q++) cam.v[q] = cam7[q];
    {
        // blackbody colours per index, made once per context
        bool fresh = c->scratch.find("r_star_colours") == c->scratch.end();
        if ((rc = c->buffer("r_star_colours", sizeof(float) * 6 * 391, &p))) return rc;
        cam.colours = (const float*)p;
        if (fresh) star_colours<<<2, 256, 0, c->stream>>>((float*)p);
    }
    GridV gv = grid_view(g);
    const dim3 blk(16, 16);
    if (v.pix_area) {
        cam.pix_area = v.pix_area;
    } else {
        if ((rc = c->buffer("r_pix_area", sizeof(float) * NP, &p))) return rc;
        cam.pix_area = (const float*)p;
        view_pixel_areas<<<grid2d(W, H), blk, 0, c->stream>>>(v.view, W, H, (float*)p);
    }
    if (!blend) {
        KTimer t(c, "pix_interp");
        pix_interp<<<grid2d(W + 1, H + 1), blk, 0, c->stream>>>(gv, g.gridlvl, v.view, W, H, f.hor, f.ver, thphi, gap);
    } else {
        GridV gb = grid_view(blend->b);
        float2* border = reinterpret_cast<float2*>(blend->border);
        {
            // findBhCenter, findBhBorders, smoothBorder x 4 (MakeImageKernel.cu:1429-1442)
            KTimer t(c, "blend_border");
            if ((rc = c->buffer("r_blend_tmp", sizeof(float2) * (2 + 2 * kAngleNum) + 64, &p))) return rc;
            float2* tmp = (float2*)p;
            int* ext = reinterpret_cast<int*>(tmp + 2 + 2 * kAngleNum);
            bh_extent_init<<<1, 64, 0, c->stream>>>(ext);
            bh_extent<<<grid2d(g.GM, g.GN), blk, 0, c->stream>>>(gv, gb, ext);
            const unsigned nb = (2 * kAngleNum + 255) / 256;
            bh_borders<<<nb, 256, 0, c->stream>>>(gv, gb, ext, border);
            smooth_border<<<nb, 256, 0, c->stream>>>(border, tmp);
            smooth_border<<<nb, 256, 0, c->stream>>>(tmp, border);
            smooth_border<<<nb, 256, 0, c->stream>>>(border, tmp);
            smooth_border<<<nb, 256, 0, c->stream>>>(tmp, border);
        }
        KTimer t(c, "pix_interp");
        pix_interp_blend<<<grid2d(W + 1, H + 1), blk, 0, c->stream>>>(gv, gb, g.gridlvl, border, blend->alpha, v.view,
                                                                      W, H, f.hor, f.ver, thphi, gap);
    }
    {
        KTimer t(c, "bh_area");
        bh_area<<<grid2d(W, H), blk, 0, c->stream>>>(thphi, W, H, bh, area, ctr, kStarCtrWords + kEnvCtrWords);
    }
    {
        KTimer t(c, "smooth");
        smooth_h<<<grid2d(W, H), blk, 0, c->stream>>>(area, gap, W, H, area_s);
        smooth_v<<<grid2d(W, H), blk, 0, c->stream>>>(area_s, gap, W, H, area);
    }
    BT_HIP(hipGetLastError());
    // The sky pass runs on the auxiliary stream beside the star pass: both
    // read the per-pixel stages made above and write their own image, and
    // each has latency-bound kernels (the lensed pixels' queues) that leave
    // the other room.  Joined before the composite.
    const bool overlap = f.star && f.map;
    uint32_t *qgroup = nullptr, *qwave = nullptr;
    unsigned* nq = nullptr;
    const float texel_size = BT_FPI / (float)s.rows;
    const SkyK sky{reinterpret_cast<const float4*>(s.table), s.rows, s.cols, texel_size, 1.0 / (double)texel_size};
    if (f.map) {
        if ((rc = c->buffer("r_env_q", sizeof(uint32_t) * 2 * (NP + 64), &p))) return rc;
        qgroup = (uint32_t*)p;
        qwave = (uint32_t*)p + NP + 64;
        nq = ctr + kStarCtrWords;
    }
    // distortEnvironmentMap: pixels with few sky columns inline, those with
    // more sixteen lanes each; then the wide ones, one wave each
    auto sky_light = [&](hipStream_t es) {
        KTimer t(c, "env_map", es);
        env_map<<<grid2d(W, H), blk, 0, es>>>(thphi, bh, sky, cam, W, H, f.offset, f.lr, area, v.view, img_map, qgroup,
                                              qwave, nq);
        env_map_group<<<(unsigned)c->num_cus * 4, 256, 0, es>>>(thphi, sky, cam, W, f.offset, f.lr, area, v.view,
                                                               img_map, qgroup, nq + kCtrGroup);
    };
    auto sky_heavy = [&](hipStream_t es) {
        KTimer t(c, "env_heavy", es);
        env_map_heavy<<<(unsigned)c->num_cus * 8, 128, 0, es>>>(thphi, sky, cam, W, f.offset, f.lr, area, v.view,
                                                               img_map, qwave, nq + kCtrHeavy);
    };
    auto join = [&]() -> hipError_t {
        const hipError_t e = hipEventRecord(c->ev_join, c->aux);
        const hipError_t w = hipStreamWaitEvent(c->stream, c->ev_join, 0);
        return e != hipSuccess ? e : w;
    };
    if (overlap) {
        BT_HIP(hipEventRecord(c->ev_fork, c->stream));
        BT_HIP(hipStreamWaitEvent(c->aux, c->ev_fork, 0));
    }
    if (f.star) {
      // the star pass; on an error the streams are joined before returning
      const int src = [&]() -> int {
        const int fw = 2 * step + 1;
        if ((rc = c->buffer("r_taps", sizeof(float) * 3 * fw * fw * NP, &p))) return rc;
        float* taps = (float*)p;
        StarQueue Q;
        if ((rc = c->buffer("r_star_lens", sizeof(float) * 3 * (NP + 64), &p))) return rc;
        Q.lens = (float*)p;
        if ((rc = c->buffer("r_star_odd", sizeof(uint32_t) * (NP + 64), &p))) return rc;
        Q.odd = (uint32_t*)p;
        Q.oddc = reinterpret_cast<uint32_t*>(area_s);   // the smoothing is through with it
        if ((rc = c->buffer("r_star_q", sizeof(uint32_t) * 6 * (NP + 64), &p))) return rc;
        Q.pix = (uint32_t*)p;
        Q.cnt = Q.pix + NP + 64;
        Q.cstart = Q.cnt + NP + 64;
        Q.owner = Q.cstart + NP + 64;
        Q.nnode = Q.owner + NP + 64;
        Q.rbase = Q.nnode + NP + 64;
        Q.wide = Q.owner;   // star_wide reads it before star_assign hands out chunks
        // tree pixels are the few whose quad crosses phi = 2 pi
        Q.rcap = (unsigned)(NP / 4 + 65536);
        if ((rc = c->buffer("r_star_ranges", sizeof(int2) * (size_t)Q.rcap, &p))) return rc;
        Q.ranges = (int2*)p;
        Q.ctr = ctr;
        if ((rc = c->buffer("r_star_lit", NP, &p))) return rc;
        Q.lit = (uint8_t*)p;
        const int NT = fw * fw * 3;
        // chunk indices beyond cap are never used: a pixel whose chunks do
        // not fit is traced by one lane in star_few
        Q.cap = (unsigned)(NP + 64);
        if ((rc = c->buffer("r_star_part", sizeof(float) * NT * (size_t)Q.cap, &p))) return rc;
        Q.partial = (float*)p;
        const unsigned nwave = (unsigned)c->num_cus * 16, nred = (unsigned)c->num_cus * 4;
        // The odd pixels' chunks and the one-lane pixels (few, long chains) run
        // beside the chunks, on the auxiliary stream once the sky pass is
        // through; from four million pixels on, where the sky pass is the
        // longer one, the one-lane pixels stay on the main stream (frames of
        // three grids, us, on the main stream and on the auxiliary one:
        // 3840x2160 1151, 1716, 1311 and 1216, 1671, 1371, 2880x1620 831, 1238,
        // 965 and 831, 1194, 1050, 2560x1440 786, 1201, 892 and 777, 1169, 962,
        // 1920x1080 587, 860, 647 and 591, 842, 638).
        // Trails fill the auxiliary stream: the odd chunks stay on the main one
        // too then.
        const bool few_on_main = !overlap || tf || NP >= (size_t(1) << 22);
        const unsigned ntree = (unsigned)c->num_cus * 4;
        const int tiles = NP >= (size_t(1) << 20) ? kScanTiles : 1;
        const dim3 gscan((unsigned)((W + 16 * tiles - 1) / (16 * tiles)), (unsigned)((H + 15) / 16));
        if (tf) {
            // with both passes on, the trails are made on the auxiliary
            // stream, their images once the pixels are sorted; the main stream
            // waits for that one before star_sum reads them
            const hipStream_t ts = overlap ? c->aux : c->stream;
            KTimer t(c, "trails", ts);
            const TrailK& T = tf->k;
            trail_clear<<<(unsigned)c->num_cus * 4, 256, 0, ts>>>(T, tf->first ? 1 : 0, 3 * NP);
            trail_grad<<<grid2d(W + 1, H + 1), blk, 0, ts>>>(thphi, W, H, T.grad);
            BT_HIP(hipGetLastError());
        }
        if (overlap) {
            sky_light(c->aux);
            sky_heavy(c->aux);
        }
        const auto trail_images = [&](hipStream_t ts) {
            KTimer t(c, "trail_images", ts);
            const TrailK& T = tf->k;
            const int span = std::max(256, few_span(NP) / 4);
            trail_hits<<<(unsigned)((NP + span - 1) / span), 256, 0, ts>>>(thphi, s, cam, W, H, f.offset, T, Q.lit,
                                                                           span);
            trail_queued<<<(unsigned)c->num_cus * 4, 256, 0, ts>>>(thphi, s, cam, W, f.offset, T, Q);
            trail_over<<<(unsigned)c->num_cus, 256, 0, ts>>>(T);
            const unsigned ncache = (unsigned)((T.S + 255) / 256);
            trail_lines<<<ncache + (unsigned)(((size_t)T.S * kTrailHits + 255) / 256), 256, 0, ts>>>(
                thphi, s, T, cam, W, H, f.offset, f.lr, area, v.view, ncache);
        };
#define BT_STAR_LAUNCH(S)                                                                                    \
    {                                                                                                       \
        {                                                                                                   \
            KTimer t(c, "star_light");                                                                      \
            star_scan<<<gscan, blk, 0, c->stream>>>(thphi, bh, s, cam, W, H, f.offset, Q, tiles);               \
        }                                                                                                   \
        KTimer t(c, "star_heavy");                                                                          \
        {                                                                                                   \
            KTimer t1(c, "star_tree");                                                                      \
            star_wide<<<nred * 2 + ntree, 64, 0, c->stream>>> (thphi, s, cam, W, H, f.offset, Q, ntree);    \
            star_assign<<<nred, 256, 0, c->stream>>>(thphi, s, cam, W, H, f.offset, f.lr, area, v.view, Q); \
            star_heads<(2 * S + 1) * (2 * S + 1) * 3><<<nred, 256, 0, c->stream>>>(thphi, cam, W, f.offset, Q); \
        }                                                                                                   \
        const hipStream_t rs = overlap ? c->aux : c->stream;                                                \
        if (overlap) {                                                                                      \
            BT_HIP(hipEventRecord(c->ev_hand, c->stream));                                                  \
            BT_HIP(hipStreamWaitEvent(rs, c->ev_hand, 0));                                                  \
        }                                                                                                   \
        {                                                                                                   \
            KTimer t2(c, "star_chunk");                                                                     \
            star_map_chunk<S, false><<<nwave, 256, 0, c->stream>>>(s, cam, taps, Q);                        \
        }                                                                                                   \
        if (tf) trail_images(rs);                                                                           \
        star_map_chunk<S, true><<<nred, 256, 0, tf ? c->stream : rs>>>(s, cam, taps, Q);                    \
        star_rest<S>(c, few_on_main ? c->stream : rs, thphi, bh, s, cam, W, H, f, area, v.view, taps, Q);   \
        if (overlap) {                                                                                      \
            BT_HIP(hipEventRecord(c->ev_back, rs));                                                         \
            BT_HIP(hipStreamWaitEvent(c->stream, c->ev_back, 0));                                           \
        }                                                                                                   \
        KTimer t3(c, "star_reduce");                                                                        \
        star_chunk_reduce<S><<<nwave, 256, 0, c->stream>>>(taps, Q);                                        \
    }
        if (step == 1)
            BT_STAR_LAUNCH(1)
        else if (step == 2)
            BT_STAR_LAUNCH(2)
        else
            BT_STAR_LAUNCH(3)
#undef BT_STAR_LAUNCH
        BT_HIP(hipGetLastError());
        const bool diffract = tf && tf->sprite;
        float* light = nullptr;
        if (diffract) {
            if ((rc = c->buffer("r_diff_light", sizeof(float) * 3 * NP, &p))) return rc;
            light = (float*)p;
        }
        {
            KTimer t(c, "star_sum");
            float* ostar = diffract ? light : (dbg ? dbg->star : nullptr);
            const float* trail = tf ? tf->k.trail : nullptr;
            if (step == 1)
                star_sum<1><<<grid2d(W, H), blk, 0, c->stream>>>(taps, Q.lit, W, H, img_star, ostar, trail);
            else if (step == 2)
                star_sum<2><<<grid2d(W, H), blk, 0, c->stream>>>(taps, Q.lit, W, H, img_star, ostar, trail);
            else
                star_sum<3><<<grid2d(W, H), blk, 0, c->stream>>>(taps, Q.lit, W, H, img_star, ostar, trail);
        }
        BT_HIP(hipGetLastError());
        if (diffract) {
            KTimer t(c, "diffraction");
            const size_t nleft = (size_t)H * ((W + kDiffCols - 1) / kDiffCols + 1), npad = (size_t)tf->fs + 2 * kDiffPad;
            if ((rc = c->buffer("r_diff_rows", sizeof(uint32_t) * (4 * NP + nleft + npad * npad), &p))) return rc;
            uint32_t* cols = (uint32_t*)p;
            float* scaled = reinterpret_cast<float*>(cols + NP);
            int* left = reinterpret_cast<int*>(cols + 4 * NP);
            uint32_t* sprite4 = cols + 4 * NP + nleft;
            diff_rows<<<(unsigned)((H + 3) / 4), 256, 0, c->stream>>>(light, W, H, cols, scaled, left, tf->sprite,
                                                                      tf->fs, sprite4);
            diff_gather<<<grid2d(W, H), 256, 0, c->stream>>>(light, cols, scaled, left, sprite4, tf->fs, W, H,
                                                             img_star, dbg ? dbg->star : nullptr);
            BT_HIP(hipGetLastError());
        }
        return BT_OK;
      }();
      if (src) {
          if (overlap) (void)join();
          return src;
      }
    }
    if (overlap) {
        BT_HIP(join());
    } else if (f.map) {
        sky_light(c->stream);
        sky_heavy(c->stream);
    }
    BT_HIP(hipGetLastError());
    {
        KTimer t(c, "composite");
        composite<<<(unsigned)((NP + 255) / 256), 256, 0, c->stream>>>(img_star, img_map, (int64_t)NP, f.star, f.map,
                                                                     d_out);
    }
    BT_HIP(hipGetLastError());
    if (dbg) {
        if (dbg->thphi) BT_HIP(hipMemcpyAsync(dbg->thphi, thphi, sizeof(float) * 2 * NC, hipMemcpyDeviceToDevice, c->stream));
        if (dbg->gap) BT_HIP(hipMemcpyAsync(dbg->gap, gap, sizeof(int) * NC, hipMemcpyDeviceToDevice, c->stream));
        if (dbg->bh) BT_HIP(hipMemcpyAsync(dbg->bh, bh, NP, hipMemcpyDeviceToDevice, c->stream));
        if (dbg->area) BT_HIP(hipMemcpyAsync(dbg->area, area, sizeof(float) * NP, hipMemcpyDeviceToDevice, c->stream));
    }
    return BT_OK;
}

}  // namespace bt
