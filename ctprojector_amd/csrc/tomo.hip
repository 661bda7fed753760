// Distance-driven tomosynthesis projector (z main axis, detector axes fixed to
// u = (1,0,0), v = (0,1,0)) on MI355X (gfx950): cuda/distanceDriven3D.cu,
// cuda/distanceDriven3DBoxInt.cu, cuda/distanceDriven3DBranchless.cu,
// cuda/distanceDriven3DUtils.cu of the reference.
//
// FP: one lane per detector cell; for every image plane z = iz (voxel edge in
// index space) the four edge-midpoint rays of the cell span a box whose area
// average is accumulated (IntegralBoxXY, cuda/cudaMath.cu:336-397), then scaled
// by the ray length through one slab.
// BP: one lane per voxel; for every view the voxel's four edge midpoints are
// projected onto the detector (centre-indexed, cuda/distanceDriven3DUtils.cu:45-56)
// and the area average of the pre-weighted projections over that box is
// accumulated.
//
// The reference's branchless mode evaluates the same box integrals through
// FP64 summed-area tables (a summed-area table of a piecewise-constant image is
// exactly bilinear between its nodes); here both modes evaluate the box
// integral directly.  Batch items are handled independently (the reference's
// BoxInt BP reuses batch 0 and its branchless BP pre-weights view 0 only,
// cuda/distanceDriven3DBoxInt.cu:257-259, cuda/distanceDriven3DBranchless.cu:347).
#include "common.h"
#include "runtime.h"
#include "ops.h"

#include <cmath>
#include <type_traits>

namespace ctp {

// exact integral of a piecewise-constant plane over [x1,x2]x[y1,y2] clamped to
// the plane (returns 0 for an empty box)
__device__ inline float box_xy(const float* __restrict__ p, float x1, float y1, float x2, float y2, int nx, int ny) {
    const float a = clampf(x1, 0.f, (float)nx), b = clampf(x2, 0.f, (float)nx);
    const float c = clampf(y1, 0.f, (float)ny), e = clampf(y2, 0.f, (float)ny);
    if (!(b > a) || !(e > c)) return 0.f;
    const int i1 = min((int)a, nx - 1), i2 = min((int)b, nx - 1);
    const int j1 = min((int)c, ny - 1), j2 = min((int)e, ny - 1);
    float s = 0.f;
    for (int j = j1; j <= j2; j++) {
        const float wy = fminf(e, (float)(j + 1)) - fmaxf(c, (float)j);
        float r = 0.f;
        for (int i = i1; i <= i2; i++) r = fmaf(fminf(b, (float)(i + 1)) - fmaxf(a, (float)i), p[(size_t)j * nx + i], r);
        s = fmaf(wy, r, s);
    }
    return s;
}

__device__ inline float3 ld3t(const float* p, int i) { return make_float3(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }

// Interval [a, b] (clamped to [0, n], n >= K) over K consecutive cells from
// cell e on: the overlaps w.  e is moved inwards at the row's end, so that the
// K cells exist.
template <int K>
struct Span {
    float w[K];
    int e;
    __device__ inline Span(float a, float b, int n) {
        const float f = min_f(floorf(a), (float)(n - K));
        e = (int)f;
        float edge = med3_f(f, a, b);
#pragma unroll
        for (int k = 0; k < K; k++) {
            const float next = med3_f(f + (float)(k + 1), a, b);
            w[k] = next - edge;
            edge = next;
        }
    }
};

// (Window form of the boxes: the loops of box_xy with their clamps, divisions
// and dependent loads took 122 us forward and 150 us backward at 256^2 x 48
// voxels, 9 views of 256^2 cells; the call now takes 138 instead of 300 us.
// Cells a box does not meet weigh 0 by the legacy product, whatever they hold.)
// The average of a plane (nx x ny cells) over the box [x1, x2] x [y1, y2], of
// which at most K cells per axis are met: cells loaded ahead of their use.
template <int K>
struct BoxCells {
    float q[K][K], wx[K], wy[K], inv;
    __device__ inline void load(const float* __restrict__ p, int nx, int ny, float x1, float x2, float y1, float y2) {
        typedef float vec __attribute__((ext_vector_type(K), aligned(4)));
        inv = __builtin_amdgcn_rcpf((x2 - x1) * (y2 - y1));
        const Span<K> x(med_clamp(x1, 0.f, (float)nx), med_clamp(x2, 0.f, (float)nx), nx);
        const Span<K> y(med_clamp(y1, 0.f, (float)ny), med_clamp(y2, 0.f, (float)ny), ny);
        const unsigned off = (unsigned)(y.e * nx + x.e);
#pragma unroll
        for (int j = 0; j < K; j++) {
            wx[j] = x.w[j];
            wy[j] = y.w[j];
            const vec v = *reinterpret_cast<const vec*>(p + off + (unsigned)(j * nx));
#pragma unroll
            for (int i = 0; i < K; i++) q[j][i] = v[i];
        }
    }
    __device__ inline float sum() const {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < K; j++) {
            float r = mul_legacy(wx[0], q[j][0]);
#pragma unroll
            for (int i = 1; i < K; i++) r += mul_legacy(wx[i], q[j][i]);
            const float t = mul_legacy(wy[j], r);
            s = j == 0 ? t : s + t;
        }
        return s;
    }
};

// FP planes of a lane in the window form: K cells per axis, two planes' loads
// in flight.
template <int K>
__device__ inline float tomo_fp_planes(const float* __restrict__ img, const Grid& g, float3 s, float rx1, float rx2,
                                       float ry1, float ry2) {
    const size_t npl = (size_t)g.nx * g.ny;
    float val = 0.f;
    auto planes = [&](int iz, auto count) {
        constexpr int N = decltype(count)::value;
        BoxCells<K> B[N];
#pragma unroll
        for (int u = 0; u < N; u++) {
            const float h = (float)(iz + u) - s.z;
            const float a1 = fmaf(rx1, h, s.x), a2 = fmaf(rx2, h, s.x);
            const float b1 = fmaf(ry1, h, s.y), b2 = fmaf(ry2, h, s.y);
            B[u].load(img + (size_t)(iz + u) * npl, g.nx, g.ny, a1, a2, b1, b2);
        }
#pragma unroll
        for (int u = 0; u < N; u++) val = fmaf(B[u].sum(), B[u].inv, val);
    };
    int iz = 0;
    for (; iz + 4 <= g.nz; iz += 4) planes(iz, std::integral_constant<int, 4>{});
    for (; iz < g.nz; iz++) planes(iz, std::integral_constant<int, 1>{});
    return val;
}

__global__ __launch_bounds__(256) void tomo_fp_kernel(float* __restrict__ prj, const float* __restrict__ img,
                                                      const float* __restrict__ pdc, const float* __restrict__ psrc,
                                                      Grid g, Det d, int nview) {
    const int iu = blockIdx.x * 32 + (threadIdx.x & 31);
    const int iv = blockIdx.y * 8 + (threadIdx.x >> 5);
    const int view = blockIdx.z;
    if (iu >= d.nu || iv >= d.nv) return;
    // cuda/distanceDriven3DBoxInt.cu:56-113
    const float u = ((float)iu - d.off_u - (d.nu - 1) / 2.0f) * d.du;
    const float v = ((float)iv - d.off_v - (d.nv - 1) / 2.0f) * d.dv;
    const float3 C = ld3t(pdc, view);
    const float3 S = ld3t(psrc, view);
    auto toimg = [&](float3 p) {
        return make_float3((p.x - g.cx) / g.dx + g.nx / 2.0f, (p.y - g.cy) / g.dy + g.ny / 2.0f,
                           (p.z - g.cz) / g.dz + g.nz / 2.0f);
    };
    float3 x1 = toimg(make_float3(C.x + u - d.du / 2, C.y + v, C.z));
    float3 x2 = toimg(make_float3(C.x + u + d.du / 2, C.y + v, C.z));
    float3 y1 = toimg(make_float3(C.x + u, C.y + v - d.dv / 2, C.z));
    float3 y2 = toimg(make_float3(C.x + u, C.y + v + d.dv / 2, C.z));
    const float3 s = toimg(S);
    if (x1.x > x2.x) { const float3 t = x1; x1 = x2; x2 = t; }
    if (y1.y > y2.y) { const float3 t = y1; y1 = y2; y2 = t; }
    const float rx1 = (x1.x - s.x) / (x1.z - s.z), rx2 = (x2.x - s.x) / (x2.z - s.z);
    const float ry1 = (y1.y - s.y) / (y1.z - s.z), ry2 = (y2.y - s.y) / (y2.z - s.z);
    // the boxes' sides are linear in the plane: the end planes' bound them
    float side = 0.f, least = 3.0e38f;
    for (int k = 0; k < 2; k++) {
        const float h = (k == 0 ? 0.f : (float)(g.nz - 1)) - s.z;
        const float w = fmaf(rx2, h, s.x) - fmaf(rx1, h, s.x), v = fmaf(ry2, h, s.y) - fmaf(ry1, h, s.y);
        side = fmaxf(side, fmaxf(w, v));
        least = fminf(least, fminf(w, v));
    }
    // (sides of no or negative length, a source within the volume's planes, stay with the loops)
    const int cells = g.nx < 3 || g.ny < 3 || __any(!(least > 1e-6f)) ? 0
                      : !__any(!(side < 0.999f))                    ? 2
                      : !__any(!(side < 1.999f))                    ? 3
                                                                    : 0;   // uniform
    float val = 0.f;
    const size_t npl = (size_t)g.nx * g.ny;
    if (cells == 2) val = tomo_fp_planes<2>(img, g, s, rx1, rx2, ry1, ry2);
    else if (cells == 3) val = tomo_fp_planes<3>(img, g, s, rx1, rx2, ry1, ry2);
    else
        for (int iz = 0; iz < g.nz; iz++) {
            const float h = (float)iz - s.z;
            const float a1 = fmaf(rx1, h, s.x), a2 = fmaf(rx2, h, s.x);
            const float b1 = fmaf(ry1, h, s.y), b2 = fmaf(ry2, h, s.y);
            val += box_xy(img + iz * npl, a1, b1, a2, b2, g.nx, g.ny) / ((a2 - a1) * (b2 - b1));
        }
    const float3 D = make_float3(C.x + u, C.y + v, C.z);
    val *= g.dz / fabsf(S.z - D.z) *
           sqrtf((S.z - D.z) * (S.z - D.z) + (S.y - D.y) * (S.y - D.y) + (S.x - D.x) * (S.x - D.x));
    prj[((size_t)view * d.nv + iv) * d.nu + iu] = val;
}

void tomo_fp(float* prj, const float* img, const float* det_center, const float* src, int B, const Grid& g,
             const Det& d, int nview, int type, hipStream_t stream) {
    (void)type;
    const size_t nimg = (size_t)g.nx * g.ny * g.nz, nprj = (size_t)d.nu * d.nv * nview;
    dim3 grid(ceil_div(d.nu, 32), ceil_div(d.nv, 8), nview), block(256);
    for (int b = 0; b < B; b++) {
        TimedLaunch t("tomo_fp", stream);
        tomo_fp_kernel<<<grid, block, 0, stream>>>(prj + b * nprj, img + b * nimg, det_center, src, g, d, nview);
        CTP_LAUNCH_CHECK();
    }
}

// PreweightBPCartKernelXY, cuda/distanceDriven3DUtils.cu:10-40
__global__ __launch_bounds__(256) void tomo_preweight_kernel(float* __restrict__ w, const float* __restrict__ prj,
                                                             const float* __restrict__ pdc, const float* __restrict__ psrc,
                                                             float dz, Det d, int nview) {
    const long n = (long)d.nu * d.nv * nview;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int iu = (int)(i % d.nu);
    const int iv = (int)((i / d.nu) % d.nv);
    const int view = (int)(i / ((long)d.nu * d.nv));
    const float u = ((float)iu - d.off_u - (d.nu - 1) / 2.0f) * d.du;
    const float v = ((float)iv - d.off_v - (d.nv - 1) / 2.0f) * d.dv;
    const float3 C = ld3t(pdc, view), S = ld3t(psrc, view);
    const float3 D = make_float3(C.x + u, C.y + v, C.z);
    w[i] = prj[i] * (dz / fabsf(S.z - D.z) *
                     sqrtf((S.z - D.z) * (S.z - D.z) + (S.y - D.y) * (S.y - D.y) + (S.x - D.x) * (S.x - D.x)));
}

__global__ __launch_bounds__(256) void tomo_bp_kernel(float* __restrict__ img, const float* __restrict__ w,
                                                      const float* __restrict__ pdc, const float* __restrict__ psrc,
                                                      Grid g, Det d, int nview) {
    const int ix = blockIdx.x * 32 + (threadIdx.x & 31);
    const int iy = blockIdx.y * 8 + (threadIdx.x >> 5);
    const int iz = blockIdx.z;
    if (ix >= g.nx || iy >= g.ny) return;
    // voxel centre, cuda/distanceDriven3DBoxInt.cu:191-193
    const float x = ((float)ix - (g.nx - 1) / 2.0f) * g.dx + g.cx;
    const float y = ((float)iy - (g.ny - 1) / 2.0f) * g.dy + g.cy;
    const float z = ((float)iz - (g.nz - 1) / 2.0f) * g.dz + g.cz;
    const float ou = d.off_u + (d.nu - 1) / 2.0f, ov = d.off_v + (d.nv - 1) / 2.0f;
    const size_t nuv = (size_t)d.nu * d.nv;
    const float rdu = 1.f / d.du, rdv = 1.f / d.dv;
    float val = 0.f;
    // shadow of the voxel on view's detector, ProjectConeToDetCart, cuda/distanceDriven3DUtils.cu:45-56
    // (the magnification, its divisions and the offsets are the same in every lane)
    auto shadow = [&](int view, float& u1, float& u2, float& v1, float& v2) {
        const float Sx = const_load(psrc, 3L * view), Sy = const_load(psrc, 3L * view + 1);
        const float Sz = const_load(psrc, 3L * view + 2), Cz = const_load(pdc, 3L * view + 2);
        const float r = (Cz - Sz) / (z - Sz);
        const float tx = Sx - const_load(pdc, 3L * view), ty = Sy - const_load(pdc, 3L * view + 1);
        u1 = fmaf(fmaf(r, x - g.dx / 2 - Sx, tx), rdu, ou);
        u2 = fmaf(fmaf(r, x + g.dx / 2 - Sx, tx), rdu, ou);
        v1 = fmaf(fmaf(r, y - g.dy / 2 - Sy, ty), rdv, ov);
        v2 = fmaf(fmaf(r, y + g.dy / 2 - Sy, ty), rdv, ov);
    };
    auto batch = [&](int view, auto count) {
        constexpr int N = decltype(count)::value;
        float u1[N], u2[N], v1[N], v2[N];
        float side = 0.f, least = 3.0e38f;
#pragma unroll
        for (int k = 0; k < N; k++) {
            shadow(view + k, u1[k], u2[k], v1[k], v2[k]);
            side = fmaxf(side, fmaxf(u2[k] - u1[k], v2[k] - v1[k]));
            least = fminf(least, fminf(u2[k] - u1[k], v2[k] - v1[k]));
        }
        if (d.nu >= 3 && d.nv >= 3 && !__any(!(side < 1.999f) || !(least > 1e-6f))) {   // uniform
            BoxCells<3> B[N];
#pragma unroll
            for (int k = 0; k < N; k++) B[k].load(w + (view + k) * nuv, d.nu, d.nv, u1[k], u2[k], v1[k], v2[k]);
#pragma unroll
            for (int k = 0; k < N; k++) val = fmaf(B[k].sum(), B[k].inv, val);
        } else {
#pragma unroll
            for (int k = 0; k < N; k++)
                val += box_xy(w + (view + k) * nuv, u1[k], v1[k], u2[k], v2[k], d.nu, d.nv) /
                       ((u2[k] - u1[k]) * (v2[k] - v1[k]));
        }
    };
    int view = 0;
    for (; view + 2 <= nview; view += 2) batch(view, std::integral_constant<int, 2>{});
    for (; view < nview; view++) batch(view, std::integral_constant<int, 1>{});
    img[((size_t)iz * g.ny + iy) * g.nx + ix] = val;
}

void tomo_bp(float* img, const float* prj, const float* det_center, const float* src, int B, const Grid& g,
             const Det& d, int nview, int type, hipStream_t stream) {
    (void)type;
    const size_t nimg = (size_t)g.nx * g.ny * g.nz, nprj = (size_t)d.nu * d.nv * nview;
    Workspace& ws = workspace_for(stream);
    Plan pl;
    pl.add<float>(nprj);
    ws.reserve(pl.bytes);
    float* w = ws.take_n<float>(nprj);
    dim3 grid(ceil_div(g.nx, 32), ceil_div(g.ny, 8), g.nz), block(256);
    for (int b = 0; b < B; b++) {
        tomo_preweight_kernel<<<ceil_div((long)nprj, 256), 256, 0, stream>>>(w, prj + b * nprj, det_center, src, g.dz, d, nview);
        CTP_LAUNCH_CHECK();
        TimedLaunch t("tomo_bp", stream);
        tomo_bp_kernel<<<grid, block, 0, stream>>>(img + b * nimg, w, det_center, src, g, d, nview);
        CTP_LAUNCH_CHECK();
    }
}

}  // namespace ctp
