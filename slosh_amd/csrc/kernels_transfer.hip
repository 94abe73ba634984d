// Particle <-> grid transfers, grid update, particle update and rigid-body
// integration of one substep on gfx950.
//
//   k_p2g            one workgroup per active block: lane = associated cell,
//                    each wave accumulates its particles' contributions to one
//                    z slab of their 27-node stencils in registers and sums them
//                    into its own LDS slab tile (no atomics, LDS or global); the
//                    6x6x6 tile, the slabs summed per node, is written once to HBM. Same per-(node, particle) arithmetic as
//                    p2g_scatter_style.slang:84-148; only the summation order
//                    differs (and is fixed for a given particle order).
//   k_grid_update    one wave per block (in a workgroup of its own): node momentum = own tile + the halo
//                    parts of the 7 "-1" neighbours' tiles, then
//                    grid_update.slang:38-163 (gravity, clamp, collision
//                    cache / collide(), boundary projection).
//   k_g2p_update     one wave per 64 entries of a block: 6x6x6 node halo in the
//                    wave's LDS tile, then per primary particle g2p.slang:150-265
//                    fused with particle_update.slang:32-160. Outputs go to the other
//                    particle buffer at the particle's sorted slot, so particle
//                    storage follows the block order of the last substep.
//   k_g2p / k_particle_update  the same two stages as separate in-place
//                    kernels, used when a hook replaces or observes G2P.
//   k_rigid_update   rigid_impulses.slang:70-121.
#include <type_traits>

#include "launch.h"
#include "../../include/slosh_hip.h"

namespace {

constexpr int ASSOC[8][3] = {{0, 0, 0}, {0, 0, 1}, {0, 1, 0}, {0, 1, 1},
                             {1, 0, 0}, {1, 0, 1}, {1, 1, 0}, {1, 1, 1}};

// A new, opaque address of the kernel's argument block: what is read through it is loaded
// after that point, instead of held in scalar registers (and spilled) from the start.
template <typename T>
__device__ inline const T &late_args() {
    auto p = (const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const T *)p;
}

// ---------------------------------------------------------------------------
// Quadratic B-spline (kernel.slang:160-174).

__device__ inline void k_eval_all(float x, float *w) {
    w[0] = 0.5f * (1.5f - x) * (1.5f - x);
    w[1] = 0.75f - (x - 1.0f) * (x - 1.0f);
    w[2] = 0.5f * (x - 0.5f) * (x - 0.5f);
}

// ---------------------------------------------------------------------------
// 3x3 helpers on shader matrices stored row-major in float[9].

__device__ inline float det3(const float *a) {
#pragma clang fp contract(off)
    return a[0] * (a[4] * a[8] - a[5] * a[7]) - a[1] * (a[3] * a[8] - a[5] * a[6]) + a[2] * (a[3] * a[7] - a[4] * a[6]);
}

__device__ inline void mul3(const float *a, const float *b, float *r) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) r[i * 3 + j] = a[i * 3 + 0] * b[0 * 3 + j] + a[i * 3 + 1] * b[1 * 3 + j] + a[i * 3 + 2] * b[2 * 3 + j];
}

// mul(transpose(a), b)
__device__ inline void mul3_tn(const float *a, const float *b, float *r) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) r[i * 3 + j] = a[0 * 3 + i] * b[0 * 3 + j] + a[1 * 3 + i] * b[1 * 3 + j] + a[2 * 3 + i] * b[2 * 3 + j];
}

// 3x3 SVD: cyclic Jacobi eigen-decomposition of A^T A (Golub & Van Loan
// symmetric Schur rotations), eigenvalues sorted descending, then a Givens QR
// of A V (the layout of McAdams et al. 2011). U and V are rotations,
// sig0 >= sig1 >= |sig2| and sign(sig2) = sign(det A). T = float or double.
// Evaluated without multiply-add contraction, operation by operation as written,
// so that the FP32 instance rounds like a plain IEEE evaluation of the same steps.
template <typename T>
__device__ void svd3(const T *a, T *u, T *sig, T *v) {
#pragma clang fp contract(off)
    const T tol = sizeof(T) == 4 ? (T)1.0e-14 : (T)1.0e-30;
    T s[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) s[i][j] = a[0 * 3 + i] * a[0 * 3 + j] + a[1 * 3 + i] * a[1 * 3 + j] + a[2 * 3 + i] * a[2 * 3 + j];
    T vv[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
#pragma unroll 1
    for (int sweep = 0; sweep < 12; sweep++) {
        T off = s[0][1] * s[0][1] + s[0][2] * s[0][2] + s[1][2] * s[1][2];
        T dg = s[0][0] * s[0][0] + s[1][1] * s[1][1] + s[2][2] * s[2][2];
        if (!(off > tol * dg)) break;
#pragma unroll
        for (int e = 0; e < 3; e++) {
            const int p = e == 2 ? 1 : 0;
            const int q = e == 0 ? 1 : 2;
            T apq = s[p][q];
            if (apq == (T)0) continue;
            T theta = (s[q][q] - s[p][p]) / ((T)2 * apq);
            T t = (theta >= (T)0 ? (T)1 : (T)-1) / (fabs(theta) + sqrt(theta * theta + (T)1));
            T c = (T)1 / sqrt(t * t + (T)1);
            T sn = t * c;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                T skp = s[k][p], skq = s[k][q];
                s[k][p] = c * skp - sn * skq;
                s[k][q] = sn * skp + c * skq;
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                T spk = s[p][k], sqk = s[q][k];
                s[p][k] = c * spk - sn * sqk;
                s[q][k] = sn * spk + c * sqk;
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                T vkp = vv[k][p], vkq = vv[k][q];
                vv[k][p] = c * vkp - sn * vkq;
                vv[k][q] = sn * vkp + c * vkq;
            }
        }
    }
    T ev[3] = {s[0][0], s[1][1], s[2][2]};
#pragma unroll
    for (int pass = 0; pass < 2; pass++)
#pragma unroll
        for (int i = 0; i < 2; i++)
            if (ev[i] < ev[i + 1]) {
                T te = ev[i];
                ev[i] = ev[i + 1];
                ev[i + 1] = te;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    T tv = vv[k][i];
                    vv[k][i] = -vv[k][i + 1];
                    vv[k][i + 1] = tv;
                }
            }
    T b[3][3];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) b[i][j] = a[i * 3 + 0] * vv[0][j] + a[i * 3 + 1] * vv[1][j] + a[i * 3 + 2] * vv[2][j];
    T qm[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
#pragma unroll
    for (int e = 0; e < 3; e++) {
        const int r0 = e == 2 ? 1 : 0;
        const int r1 = e == 0 ? 1 : 2;
        const int col = r0;
        T x = b[r0][col], y = b[r1][col];
        T r = sqrt(x * x + y * y);
        T c = (T)1, sn = (T)0;
        if (r > (T)0) {
            c = x / r;
            sn = y / r;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            T b0 = b[r0][k], b1 = b[r1][k];
            b[r0][k] = c * b0 + sn * b1;
            b[r1][k] = -sn * b0 + c * b1;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            T q0 = qm[k][r0], q1 = qm[k][r1];
            qm[k][r0] = c * q0 + sn * q1;
            qm[k][r1] = -sn * q0 + c * q1;
        }
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        sig[i] = b[i][i];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            u[i * 3 + j] = qm[i][j];
            v[i * 3 + j] = vv[i][j];
        }
    }
}

// U diag(s) V^T
template <typename T>
__device__ inline void svd_recompose(const T *u, const T *s, const T *v, T *r) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) r[i * 3 + j] = (u[i * 3 + 0] * s[0]) * v[j * 3 + 0] + (u[i * 3 + 1] * s[1]) * v[j * 3 + 1] + (u[i * 3 + 2] * s[2]) * v[j * 3 + 2];
}

// ---------------------------------------------------------------------------
// Material models (shaders/slosh/models).

// neo_hookean_elasticity.slang:16-27
__device__ inline void nh_stress(float lambda, float mu, const float *f, float *st) {
#pragma clang fp contract(off)
    float j = fmaxf(det3(f), 1.0e-10f);
    float diag = lambda * logf(j) - mu;
    mul3_tn(f, f, st);
#pragma unroll
    for (int k = 0; k < 9; k++) st[k] *= mu;
    st[0] += diag;
    st[4] += diag;
    st[8] += diag;
}

// linear_elasticity.slang:135-148 (fixed-corotated)
__device__ inline void fc_stress(float lambda, float mu, const float *f, float *st) {
#pragma clang fp contract(off)
    float u[9], s[3], v[9], rc[9];
    svd3<float>(f, u, s, v);
    float j = s[0] * s[1] * s[2];
    float sm1[3] = {s[0] - 1.0f, s[1] - 1.0f, s[2] - 1.0f};
    float diag = lambda * (j - 1.0f) * j;
    svd_recompose(u, sm1, v, rc);
    mul3_tn(f, rc, st);
    float k2 = 2.0f * mu;
#pragma unroll
    for (int k = 0; k < 9; k++) st[k] *= k2;
    st[0] += diag;
    st[4] += diag;
    st[8] += diag;
}

// drucker_prager.slang:144-200: returns the projected deformation gradient in f,
// updates state = {plastic det, hardening, log volume gain}.
__device__ inline void dp_project(float *state, const float4 hp, float lambda, float mu, float *f) {
#pragma clang fp contract(off)
    if (lambda == 0.0f) return;
    float u[9], s[3], v[9];
    svd3<float>(f, u, s, v);
    float angle = hp.x + (hp.y * state[1] - hp.w) * expf(-hp.z * state[1]);
    float s_angle = sinf(angle);
    float alpha = sqrtf(2.0f / 3.0f) * (2.0f * s_angle) / (3.0f - s_angle);
    const float d = 3.0f;
    float strain[3], dev[3];
    float lvg = state[2];
#pragma unroll
    for (int i = 0; i < 3; i++) strain[i] = logf(s[i]) + lvg / d;
    float tr = strain[0] + strain[1] + strain[2];
#pragma unroll
    for (int i = 0; i < 3; i++) dev[i] = strain[i] - tr / d;
    float ns[3];
    float hard;
    if (tr > 0.0f || (dev[0] == 0.0f && dev[1] == 0.0f && dev[2] == 0.0f)) {
        ns[0] = ns[1] = ns[2] = 1.0f;
        hard = sqrtf(strain[0] * strain[0] + strain[1] * strain[1] + strain[2] * strain[2]);
    } else {
        float dn = sqrtf(dev[0] * dev[0] + dev[1] * dev[1] + dev[2] * dev[2]);
        float gamma = dn + (d * lambda + 2.0f * mu) / (2.0f * mu) * tr * alpha;
        if (gamma <= 0.0f) return;
#pragma unroll
        for (int i = 0; i < 3; i++) ns[i] = expf(strain[i] - dev[i] * (gamma / dn));
        hard = gamma;
    }
    float prev_det = s[0] * s[1] * s[2];
    float new_det = ns[0] * ns[1] * ns[2];
    state[0] = state[0] * prev_det / new_det;
    state[2] = state[2] + logf(prev_det) - logf(new_det);
    state[1] = state[1] + hard;
    svd_recompose(u, ns, v, f);
}

// Refined variants of the SVD-dependent steps. In FP32, F - R and log(sigma)
// near sigma = 1 lose ~5 digits to cancellation, which is the size of the parity
// tolerance. Here the quantities that cancel are computed to FP64 accuracy: the
// polar rotation R by FP64 Newton iterations from F; the principal directions from
// the eigen-decomposition of F^T F, less I near a rotation, and the log strains from its
// eigenvalues there or from the stretches |F v| of the directions.

// Orthogonal polar factor r of a (a = r s, s symmetric positive definite) by
// Newton's iteration x <- (g x + x^-T / g) / 2 with determinant scaling
// g = det(x)^(-1/3) while det(x) is far from 1 (N. J. Higham, "Computing the
// polar decomposition -- with applications", SIAM J. Sci. Stat. Comput. 7(4),
// 1986). For det(a) > 0 this is U V^T of the SVD a = U diag(sig) V^T. Returns
// false (r undefined) if det(a) <= 0 or it does not converge.
//
// Convergence is quadratic: a step of size d leaves an error of about d^2 / 2
// (d per entry: at most 9/2 d^2 in norm), so the step that is below 1e-8 is the
// last one (4.5e-16, round-off: the largest error of 20000 random gradients at each strain
// from 1e-7 to 0.2 is 3.3e-16, as with one more step; stopped below 3e-8 it was 1.0e-15).
// Strains of 1e-4 to 1e-2 take 2.7 to 3.6 iterations on average.
__device__ inline bool polar_f64(const float *a, double *x) {
#pragma unroll
    for (int k = 0; k < 9; k++) x[k] = a[k];
#pragma unroll 1
    for (int it = 0; it < 24; it++) {
        double c[9];
        c[0] = x[4] * x[8] - x[5] * x[7];
        c[1] = x[5] * x[6] - x[3] * x[8];
        c[2] = x[3] * x[7] - x[4] * x[6];
        c[3] = x[2] * x[7] - x[1] * x[8];
        c[4] = x[0] * x[8] - x[2] * x[6];
        c[5] = x[1] * x[6] - x[0] * x[7];
        c[6] = x[1] * x[5] - x[2] * x[4];
        c[7] = x[2] * x[3] - x[0] * x[5];
        c[8] = x[0] * x[4] - x[1] * x[3];
        const double det = x[0] * c[0] + x[1] * c[1] + x[2] * c[2];
        if (!(det > 0.0)) return false;
        // Any positive scale keeps the iteration convergent; FP32 is enough for it.
        const double g = fabs(det - 1.0) > 0.05 ? (double)(1.0f / cbrtf((float)det)) : 1.0;
        const double h = 0.5 / (g * det);
        double diff = 0.0, norm = 0.0;
#pragma unroll
        for (int k = 0; k < 9; k++) {
            const double nx = 0.5 * g * x[k] + h * c[k];
            diff = fmax(diff, fabs(nx - x[k]));
            norm = fmax(norm, fabs(nx));
            x[k] = nx;
        }
        if (diff <= 1.0e-8 * norm) return true;
    }
    return false;
}

// One Jacobi rotation in the (p, q) plane of a symmetric 3x3 matrix (its entries
// pp, qq, pq and the third row's rp, rq) and of the columns p, q of v. The angle
// only has to be near the one that annihilates pq (the sweeps converge all the
// same), so its tangent comes from FP32 approximations; the cosine is then
// corrected to FP64 by a Newton step, which keeps the rotation orthonormal.
__device__ inline void jacobi_rotate(double &pp, double &qq, double &pq, double &rp, double &rq, double *v, int p, int q) {
    const float d = (float)(qq - pp), b = 2.0f * (float)pq;
    const float den = fabsf(d) + __builtin_amdgcn_sqrtf(d * d + b * b);
    const float tf = den > 0.0f ? (d < 0.0f ? -b : b) * __builtin_amdgcn_rcpf(den) : 0.0f;
    const double t = tf, w = 1.0 + t * t;
    const double c0 = __builtin_amdgcn_rsqf((float)w);
    const double c = c0 * (1.5 - 0.5 * w * c0 * c0), s = t * c;
    const double cc = c * c, ss = s * s, cs = c * s, x = 2.0 * cs * pq, npp = cc * pp - x + ss * qq, nqq = ss * pp + x + cc * qq;
    pq = (cc - ss) * pq + cs * (pp - qq);
    pp = npp;
    qq = nqq;
    const double nrp = c * rp - s * rq;
    rq = s * rp + c * rq;
    rp = nrp;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double a = v[k * 3 + p], z = v[k * 3 + q];
        v[k * 3 + p] = c * a - s * z;
        v[k * 3 + q] = s * a + c * z;
    }
}

// Eigenvectors (the columns of v, a rotation) of F^T F by cyclic Jacobi sweeps. With
// NEAR and where F^T F is near I, true is returned and e holds its eigenvalues less 1, which then lose
// nothing to the 1. Elsewhere that difference would lose what is left of a matrix far
// smaller than I: e orders the eigenvalues only (they are scaled to a trace of 1, which
// also keeps the FP32 angles of tiny and huge gradients in range).
template <bool NEAR>
__device__ inline bool eigen_f64(const float *f32, double *e, double *v) {
    double e00, e11, e22, e01, e02, e12;
    bool near;
    {
        // The products are exact in FP64, the sums lose only FP64 round-off.
        double f[9];
#pragma unroll
        for (int k = 0; k < 9; k++) f[k] = f32[k];
        e00 = f[0] * f[0] + f[3] * f[3] + f[6] * f[6];
        e11 = f[1] * f[1] + f[4] * f[4] + f[7] * f[7];
        e22 = f[2] * f[2] + f[5] * f[5] + f[8] * f[8];
        e01 = f[0] * f[1] + f[3] * f[4] + f[6] * f[7];
        e02 = f[0] * f[2] + f[3] * f[5] + f[6] * f[8];
        e12 = f[1] * f[2] + f[4] * f[5] + f[7] * f[8];
        near = NEAR && fmax(fmax(fabs(e00 - 1.0), fabs(e11 - 1.0)), fabs(e22 - 1.0)) <= 0.5;
        if (near) {
            e00 -= 1.0;
            e11 -= 1.0;
            e22 -= 1.0;
        } else {
            const double k = 1.0 / (e00 + e11 + e22);
            e00 *= k;
            e11 *= k;
            e22 *= k;
            e01 *= k;
            e02 *= k;
            e12 *= k;
        }
    }
#pragma unroll
    for (int k = 0; k < 9; k++) v[k] = k % 4 == 0 ? 1.0 : 0.0;
#pragma unroll 1
    for (int sweep = 0; sweep < 12; sweep++) {
        const double off = e01 * e01 + e02 * e02 + e12 * e12;
        const double one = near ? 1.0 : 0.0;
        const double dg = (one + e00) * (one + e00) + (one + e11) * (one + e11) + (one + e22) * (one + e22);
        if (!(off > 1.0e-30 * dg)) break;
        jacobi_rotate(e00, e11, e01, e02, e12, v, 0, 1);
        jacobi_rotate(e00, e22, e02, e01, e12, v, 0, 2);
        jacobi_rotate(e11, e22, e12, e01, e02, v, 1, 2);
    }
    e[0] = e00;
    e[1] = e11;
    e[2] = e22;
    return near;
}

// |F v_i|^2 of column i of v.
__device__ inline double stretch2(const float *f, const double *v, int i) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double w = (double)f[3 * k] * v[i] + (double)f[3 * k + 1] * v[3 + i] + (double)f[3 * k + 2] * v[6 + i];
        s += w * w;
    }
    return s;
}

__device__ inline double det3d(const float *a) {
    const double x[9] = {a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8]};
    return x[0] * (x[4] * x[8] - x[5] * x[7]) - x[1] * (x[3] * x[8] - x[5] * x[6]) + x[2] * (x[3] * x[7] - x[4] * x[6]);
}

// U V^T of the SVD with U and V rotations, for an F with det F <= 0 or so close
// to singular that polar_f64 fails (such a particle is disabled unless its FP32
// determinant rounds to a positive value): the two larger singular values give
// their left vectors, the third is their cross product.
__device__ inline void rotation_by_eigen(const float *f, double *r) {
    double e[3], v[9];
    eigen_f64<false>(f, e, v);
    // The column of the smallest eigenvalue goes last (cyclically: v stays a rotation).
#pragma unroll 1
    for (int turn = 0; turn < 2 && (e[0] < e[2] || e[1] < e[2]); turn++) {
        const double t = e[0];
        e[0] = e[1];
        e[1] = e[2];
        e[2] = t;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double w = v[3 * k];
            v[3 * k] = v[3 * k + 1];
            v[3 * k + 1] = v[3 * k + 2];
            v[3 * k + 2] = w;
        }
    }
    double u[2][3];
#pragma unroll
    for (int j = 0; j < 2; j++) {
#pragma unroll
        for (int i = 0; i < 3; i++) u[j][i] = (double)f[3 * i] * v[j] + (double)f[3 * i + 1] * v[3 + j] + (double)f[3 * i + 2] * v[6 + j];
        const double w = 1.0 / sqrt(u[j][0] * u[j][0] + u[j][1] * u[j][1] + u[j][2] * u[j][2]);
#pragma unroll
        for (int i = 0; i < 3; i++) u[j][i] *= w;
    }
    const double c[3] = {u[0][1] * u[1][2] - u[0][2] * u[1][1], u[0][2] * u[1][0] - u[0][0] * u[1][2],
                         u[0][0] * u[1][1] - u[0][1] * u[1][0]};
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) r[3 * i + j] = u[0][i] * v[3 * j] + u[1][i] * v[3 * j + 1] + c[i] * v[3 * j + 2];
}

// linear_elasticity.slang:135-148 in FP64: tau = 2 mu (F - R) F^T + lambda (J - 1) J I
// with R the polar rotation (U V^T of the SVD), J = det F. tau is symmetric: six entries.
__device__ inline void fc_stress_f64(float lambda, float mu, const float *f32, float *st) {
    double r[9];
    if (!polar_f64(f32, r)) rotation_by_eigen(f32, r);
    double f[9];
#pragma unroll
    for (int k = 0; k < 9; k++) {
        f[k] = f32[k];
        r[k] = f[k] - r[k];
    }
    const double j = f[0] * (f[4] * f[8] - f[5] * f[7]) - f[1] * (f[3] * f[8] - f[5] * f[6]) + f[2] * (f[3] * f[7] - f[4] * f[6]);
    const double mu2 = 2.0 * (double)mu, vol = (double)lambda * (j - 1.0) * j;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int k = i; k < 3; k++) {
            double r2 = mu2 * (f[0 * 3 + i] * r[0 * 3 + k] + f[1 * 3 + i] * r[1 * 3 + k] + f[2 * 3 + i] * r[2 * 3 + k]);
            if (i == k) r2 += vol;
            st[i * 3 + k] = (float)r2;
            if (i != k) st[k * 3 + i] = (float)r2;
        }
}

// log(1 + e) / 2, the log of a singular value from the eigenvalue 1 + e of
// F^T F, for |e| <= 1/4: atanh(e / (2 + e)) by its series (relative error below
// 1e-10).
__device__ inline double half_log1p(double e) {
    const double r = e / (2.0 + e), q = r * r;
    return r + r * q * (1.0 / 3.0 + q * (1.0 / 5.0 + q * (1.0 / 7.0 + q * (1.0 / 9.0 + q * (1.0 / 11.0)))));
}

// exp(x) - 1: its Taylor series for |x| <= 1/4 (relative error below 5e-11), the
// library's function beyond.
__device__ inline double exp_m1(double x) {
    if (fabs(x) <= 0.25) {
        double p = 1.0 / 40320.0;
        p = 1.0 / 5040.0 + x * p;
        p = 1.0 / 720.0 + x * p;
        p = 1.0 / 120.0 + x * p;
        p = 1.0 / 24.0 + x * p;
        p = 1.0 / 6.0 + x * p;
        p = 0.5 + x * p;
        return x + x * x * p;
    }
    return expm1(x);
}

// drucker_prager.slang:144-200 (Klar et al. 2016 return mapping in log-strain
// space on the singular values), refined as described above. The projected
// gradient is U diag(s') V^T = F V diag(s' / s) V^T, so only V and the ratios
// s' / s - 1 = exp(log s' - log s) - 1 are needed, and F changes by the small
// product F V diag(s' / s - 1) V^T.
//
// VALU-bound: 4 sweeps of 3 rotations (~50 FP64 operations each) take the place
// of an FP32 SVD, its FP64 refinement and FP32 logarithms (~3000 operations).
__device__ inline void dp_project_f64(float *state, const float4 hp, float lambda_f, float mu_f, float *f32) {
    if (lambda_f == 0.0f) return;
    if (!(det3d(f32) > 0.0)) {
        // The log of a singular value that is not positive is NaN, as in the shader;
        // the particle is disabled by the update.
        const float nan = __uint_as_float(0x7fc00000u);
        state[0] = state[1] = state[2] = nan;
#pragma unroll
        for (int k = 0; k < 9; k++) f32[k] = nan;
        return;
    }
    double e[3], v[9];
    const bool near = eigen_f64<true>(f32, e, v);
    const float q = state[1];
    const float angle = hp.x + (hp.y * q - hp.w) * expf(-hp.z * q);
    const float sa = sinf(angle);
    const double alpha = (double)(sqrtf(2.0f / 3.0f) * (2.0f * sa) / (3.0f - sa));
    const double lambda = lambda_f, mu = mu_f, third = (double)state[2] / 3.0;
    // The log of a singular value: beyond the series' range from the stretch of its
    // direction, whose square keeps the digits that an eigenvalue far below the largest one
    // (1e-16 of that one off) has lost.
    double raw[3], dev[3];
#pragma unroll
    for (int i = 0; i < 3; i++)
        raw[i] = (near & (fabs(e[i]) <= 0.25)) ? half_log1p(e[i]) : 0.5 * log(stretch2(f32, v, i));
    const double tr = raw[0] + raw[1] + raw[2] + 3.0 * third;
#pragma unroll
    for (int i = 0; i < 3; i++) dev[i] = raw[i] + third - tr / 3.0;
    // Tension (s' = 1: F becomes its polar rotation) or the projection onto the cone,
    // selected without branches: one gave a wrong register to the lanes that reach
    // the first case through its second condition.
    const bool tension = (tr > 0.0) | ((dev[0] == 0.0) & (dev[1] == 0.0) & (dev[2] == 0.0));
    const double dn = sqrt(dev[0] * dev[0] + dev[1] * dev[1] + dev[2] * dev[2]);
    const double gamma = dn + (3.0 * lambda + 2.0 * mu) / (2.0 * mu) * tr * alpha;
    if (!tension & (gamma <= 0.0)) return;
    const double k = gamma / (tension ? 1.0 : dn);
    // log s' - log s per direction
    double dl[3], n2 = 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        n2 += (raw[i] + third) * (raw[i] + third);
        dl[i] = tension ? -raw[i] : third - dev[i] * k;
    }
    const double hard = tension ? sqrt(n2) : gamma;
    const double r0 = exp_m1(dl[0]), r1 = exp_m1(dl[1]), r2 = exp_m1(dl[2]);
    state[0] = (float)((double)state[0] / ((1.0 + r0) * (1.0 + r1) * (1.0 + r2)));
    state[2] = (float)((double)state[2] - (dl[0] + dl[1] + dl[2]));
    state[1] = (float)((double)state[1] + hard);
    double m[9];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = i; j < 3; j++)
            m[i * 3 + j] = m[j * 3 + i] = r0 * v[i * 3] * v[j * 3] + r1 * v[i * 3 + 1] * v[j * 3 + 1] + r2 * v[i * 3 + 2] * v[j * 3 + 2];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const double row[3] = {f32[i * 3], f32[i * 3 + 1], f32[i * 3 + 2]};
#pragma unroll
        for (int j = 0; j < 3; j++)
            f32[i * 3 + j] = (float)(row[j] + (row[0] * m[j] + row[1] * m[3 + j] + row[2] * m[6 + j]));
    }
}

// ---------------------------------------------------------------------------
// Shapes, poses and collisions (shaders/slosh/rbd, shaders/slosh/collision).
//
// The contact geometry is evaluated without FMA contraction, with the operation
// order of plain IEEE single precision. A contact normal is (projection - node) /
// distance, so for a node near a surface its rounding error grows as 1 / distance:
// contracting some products (the compiler's default) moves such normals by up to
// 1e-4, where the uncontracted evaluation reproduces the CPU's bits.

__device__ inline float3 quat_rotate(float4 q, float3 v) {
#pragma clang fp contract(off)
    float3 t = make_float3(2.0f * (q.y * v.z - q.z * v.y), 2.0f * (q.z * v.x - q.x * v.z), 2.0f * (q.x * v.y - q.y * v.x));
    return make_float3(v.x + q.w * t.x + (q.y * t.z - q.z * t.y), v.y + q.w * t.y + (q.z * t.x - q.x * t.z),
                       v.z + q.w * t.z + (q.x * t.y - q.y * t.x));
}

// Sim3 (quaternion, translation, uniform scale) point transforms.
__device__ inline float3 sim_mul_pt(float4 rot, float4 ts, float3 p) {
#pragma clang fp contract(off)
    float3 r = quat_rotate(rot, make_float3(p.x * ts.w, p.y * ts.w, p.z * ts.w));
    return make_float3(r.x + ts.x, r.y + ts.y, r.z + ts.z);
}
__device__ inline float3 sim_inv_mul_pt(float4 rot, float4 ts, float3 p) {
#pragma clang fp contract(off)
    float3 r = quat_rotate(make_float4(-rot.x, -rot.y, -rot.z, rot.w), make_float3(p.x - ts.x, p.y - ts.y, p.z - ts.z));
    return make_float3(r.x / ts.w, r.y / ts.w, r.z / ts.w);
}

__device__ inline float sgn(float x) { return x > 0.0f ? 1.0f : (x < 0.0f ? -1.0f : 0.0f); }

// cuboid.slang:34-63
__device__ inline bool cuboid_project_boundary(float3 he, float3 pt, float3 *out) {
#pragma clang fp contract(off)
    float3 op;
    op.x = pt.x + (fmaxf(-he.x - pt.x, 0.0f) - fmaxf(pt.x - he.x, 0.0f));
    op.y = pt.y + (fmaxf(-he.y - pt.y, 0.0f) - fmaxf(pt.y - he.y, 0.0f));
    op.z = pt.z + (fmaxf(-he.z - pt.z, 0.0f) - fmaxf(pt.z - he.z, 0.0f));
    float sx = sgn(pt.x), sy = sgn(pt.y), sz = sgn(pt.z);
    sx = sx + (fabsf(sx) - 1.0f);
    sy = sy + (fabsf(sy) - 1.0f);
    sz = sz + (fabsf(sz) - 1.0f);
    float dx = he.x - sx * pt.x, dy = he.y - sy * pt.y, dz = he.z - sz * pt.z;
    bool pick_x = dx <= dy && dx <= dz;
    bool pick_y = dy <= dx && dy <= dz;
    float3 ip = pt;
    if (pick_x) ip.x = pt.x + dx * sx;
    else if (pick_y) ip.y = pt.y + dy * sy;
    else ip.z = pt.z + dz * sz;
    bool inside = pt.x == op.x && pt.y == op.y && pt.z == op.z;
    *out = inside ? ip : op;
    return inside;
}

// ball.slang:39-50
__device__ inline bool ball_project_boundary(float radius, float3 pt, float3 *out) {
#pragma clang fp contract(off)
    float dist = sqrtf(pt.x * pt.x + pt.y * pt.y + pt.z * pt.z);
    if (dist != 0.0f) {
        float k = radius / dist;
        *out = make_float3(pt.x * k, pt.y * k, pt.z * k);
    } else {
        *out = make_float3(0.0f, radius, 0.0f);
    }
    return dist <= radius;
}

// segment.slang:10-28: closest point of segment [a, b] to p.
__device__ inline float3 segment_project(float3 a, float3 b, float3 p) {
#pragma clang fp contract(off)
    const float3 ab = make_float3(b.x - a.x, b.y - a.y, b.z - a.z);
    const float3 ap = make_float3(p.x - a.x, p.y - a.y, p.z - a.z);
    const float ab_ap = ab.x * ap.x + ab.y * ap.y + ab.z * ap.z;
    const float sqnab = ab.x * ab.x + ab.y * ab.y + ab.z * ab.z;
    if (ab_ap <= 0.0f) return a;
    if (ab_ap >= sqnab) return b;
    const float u = ab_ap / sqnab;
    return make_float3(a.x + ab.x * u, a.y + ab.y * u, a.z + ab.z * u);
}

// capsule.slang:41-58 and 77-100 (segment a..b, radius r).
__device__ inline bool capsule_project_boundary(float3 a, float3 b, float r, float3 pt, float3 *out) {
#pragma clang fp contract(off)
    const float3 on_axis = segment_project(a, b, pt);
    const float3 d = make_float3(pt.x - on_axis.x, pt.y - on_axis.y, pt.z - on_axis.z);
    const float dist = sqrtf(d.x * d.x + d.y * d.y + d.z * d.z);
    if (dist > 0.0f) {
        const float k = r / dist;
        *out = make_float3(on_axis.x + d.x * k, on_axis.y + d.y * k, on_axis.z + d.z * k);
        return dist <= r;
    }
    // On the axis: the first vector of the orthonormal basis of the axis direction.
    float3 ax = make_float3(b.x - a.x, b.y - a.y, b.z - a.z);
    const float len = sqrtf(ax.x * ax.x + ax.y * ax.y + ax.z * ax.z);
    ax = make_float3(ax.x / len, ax.y / len, ax.z / len);
    const float sign = ax.z >= 0.0f ? 1.0f : -1.0f;
    const float ka = -1.0f / (sign + ax.z);
    const float kb = ax.x * ax.y * ka;
    const float3 dir = make_float3(1.0f + sign * ax.x * ax.x * ka, sign * kb, -sign * ax.x);
    *out = make_float3(on_axis.x + dir.x * r, on_axis.y + dir.y * r, on_axis.z + dir.z * r);
    return true;
}

// |(x, z)| and the unit direction of (x, z) from the y axis ((1, 0) on the axis).
__device__ inline float planar_dir(float3 pt, float *dx, float *dz) {
#pragma clang fp contract(off)
    const float pd = sqrtf(pt.x * pt.x + pt.z * pt.z);
    *dx = pd > 0.0f ? pt.x / pd : 1.0f;
    *dz = pd > 0.0f ? pt.z / pd : 0.0f;
    return pd;
}

// cylinder.slang:68-128 (axis y, half height hh, radius r).
__device__ inline bool cylinder_project_boundary(float hh, float r, float3 pt, float3 *out) {
#pragma clang fp contract(off)
    float dx, dz;
    const float pd = planar_dir(pt, &dx, &dz);
    const float px = dx * r, pz = dz * r;
    if (pt.y >= -hh && pt.y <= hh && pd <= r) {
        const float to_top = hh - pt.y, to_bottom = pt.y - (-hh), to_side = r - pd;
        if (to_top < to_bottom && to_top < to_side) *out = make_float3(pt.x, hh, pt.z);
        else if (to_bottom < to_top && to_bottom < to_side) *out = make_float3(pt.x, -hh, pt.z);
        else *out = make_float3(px, pt.y, pz);
        return true;
    }
    if (pt.y > hh || pt.y < -hh) {
        const float y = pt.y > hh ? hh : -hh;
        *out = pd <= r ? make_float3(pt.x, y, pt.z) : make_float3(px, y, pz);
    } else {
        *out = make_float3(px, pt.y, pz);
    }
    return false;
}

__device__ inline float3 cross3f(float3 a, float3 b) {
#pragma clang fp contract(off)
    return make_float3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}

// cone.slang:61-120 (axis y, apex at +hh, base disc of radius r at -hh).
__device__ inline bool cone_project_boundary(float hh, float r, float3 pt, float3 *out) {
#pragma clang fp contract(off)
    float dx, dz;
    const float pd = planar_dir(pt, &dx, &dz);
    const float3 on_base = make_float3(pt.x, -hh, pt.z);
    if (pt.y < -hh && pd <= r) {
        *out = on_base;
        return false;
    }
    const float3 rim = make_float3(dx * r, -hh, dz * r);
    const float3 apex = make_float3(0.0f, hh, 0.0f);
    const float3 side = make_float3(rim.x - apex.x, rim.y - apex.y, rim.z - apex.z);
    const float3 proj = segment_project(apex, rim, pt);
    const float3 c1 = cross3f(side, make_float3(pt.x - apex.x, pt.y - apex.y, pt.z - apex.z));
    const float3 c2 = cross3f(side, make_float3(0.0f, -2.0f * hh, 0.0f));
    if (pt.y >= -hh && pt.y <= hh && c1.x * c2.x + c1.y * c2.y + c1.z * c2.z >= 0.0f) {
        const float3 tp = make_float3(proj.x - pt.x, proj.y - pt.y, proj.z - pt.z);
        const float3 tb = make_float3(on_base.x - pt.x, on_base.y - pt.y, on_base.z - pt.z);
        *out = (tp.x * tp.x + tp.y * tp.y + tp.z * tp.z > tb.x * tb.x + tb.y * tb.y + tb.z * tb.z) ? on_base : proj;
        return true;
    }
    *out = proj;
    return false;
}

struct Colliders {
    const float4 *shapes; // 2 per body: a, b
    const float4 *poses;  // 2 per body: rotation, translation_scale
    const uint2 *mats;    // (type, friction bits)
    uint32_t count;
    const float4 *mesh_vtx;   // trimesh collision vertices: BVH AABBs, vertices, pseudo-normals
    const uint32_t *mesh_idx; // trimesh collision indices: BVH topology, triangles
    // The BVHs of the trimesh bodies as the walk reads them (see k_pack_mesh), each
    // body's first node, and how its closest triangles are found (MESH_*).
    const float4 *mesh_nodes, *mesh_leaves;
    const uint32_t *mesh_base, *mesh_search;
    const float *mesh_size;  // largest coordinate
};

// triangle_project_local_point_and_get_location (trimesh.slang:304-377): closest
// point of triangle (a, b, c) to p; feature 0 = vertex (id 0..2 = a, b, c),
// 1 = edge (id 0 = ab, 1 = bc, 2 = ca), 2 = face, 3 = degenerate (the point itself).
__device__ inline float3 triangle_project(float3 a, float3 b, float3 c, float3 p, uint32_t *feat, uint32_t *id) {
#pragma clang fp contract(off)
    const float3 ab = make_float3(b.x - a.x, b.y - a.y, b.z - a.z);
    const float3 ac = make_float3(c.x - a.x, c.y - a.y, c.z - a.z);
    const float3 ap = make_float3(p.x - a.x, p.y - a.y, p.z - a.z);
    auto dot = [](float3 u, float3 v) { return u.x * v.x + u.y * v.y + u.z * v.z; };
    const float ab_ap = dot(ab, ap), ac_ap = dot(ac, ap);
    if (ab_ap <= 0.0f && ac_ap <= 0.0f) {
        *feat = 0u; *id = 0u;
        return a;
    }
    const float3 bp = make_float3(p.x - b.x, p.y - b.y, p.z - b.z);
    const float ab_bp = dot(ab, bp), ac_bp = dot(ac, bp);
    if (ab_bp >= 0.0f && ac_bp <= ab_bp) {
        *feat = 0u; *id = 1u;
        return b;
    }
    const float3 cp = make_float3(p.x - c.x, p.y - c.y, p.z - c.z);
    const float ab_cp = dot(ab, cp), ac_cp = dot(ac, cp);
    if (ac_cp >= 0.0f && ab_cp <= ac_cp) {
        *feat = 0u; *id = 2u;
        return c;
    }
    const float3 bc = make_float3(c.x - b.x, c.y - b.y, c.z - b.z);
    // stable_check_edges_voronoi (trimesh.slang:257-302)
    const float3 n = cross3f(ab, ac);
    const float vc = dot(n, cross3f(ab, ap));
    if (vc < 0.0f && ab_ap >= 0.0f && ab_bp <= 0.0f) {
        const float v = ab_ap / dot(ab, ab);
        *feat = 1u; *id = 0u;
        return make_float3(a.x + ab.x * v, a.y + ab.y * v, a.z + ab.z * v);
    }
    const float vb = -dot(n, cross3f(ac, cp));
    if (vb < 0.0f && ac_ap >= 0.0f && ac_cp <= 0.0f) {
        const float w = ac_ap / dot(ac, ac);
        *feat = 1u; *id = 2u;
        return make_float3(a.x + ac.x * w, a.y + ac.y * w, a.z + ac.z * w);
    }
    const float va = dot(n, cross3f(bc, bp));
    if (va < 0.0f && ac_bp - ab_bp >= 0.0f && ab_cp - ac_cp >= 0.0f) {
        const float w = dot(bc, bp) / dot(bc, bc);
        *feat = 1u; *id = 1u;
        return make_float3(b.x + bc.x * w, b.y + bc.y * w, b.z + bc.z * w);
    }
    if (va + vb + vc != 0.0f) {
        const float denom = 1.0f / (va + vb + vc);
        const float v = vb * denom, w = vc * denom;
        *feat = 2u; *id = 0u;
        return make_float3(a.x + ab.x * v + ac.x * w, a.y + ab.y * v + ac.y * w, a.z + ab.z * v + ac.z * w);
    }
    *feat = 3u; *id = 0u;
    return p;
}

// Distance of a point from a box (0 inside), in the operation order of the BVH walk.
__device__ inline float box_distance(float4 mn, float4 mx, float3 pt) {
#pragma clang fp contract(off)
    const float qx = (pt.x + (fmaxf(mn.x - pt.x, 0.0f) - fmaxf(pt.x - mx.x, 0.0f))) - pt.x;
    const float qy = (pt.y + (fmaxf(mn.y - pt.y, 0.0f) - fmaxf(pt.y - mx.y, 0.0f))) - pt.y;
    const float qz = (pt.z + (fmaxf(mn.z - pt.z, 0.0f) - fmaxf(pt.z - mx.z, 0.0f))) - pt.z;
    return sqrtf(qx * qx + qy * qy + qz * qz);
}

// The closest point of the triangle of BVH leaf `leaf` (3 vertices, the triangle
// index in the first one's w), its distance and the feature it lies on.
__device__ inline float leaf_distance(const float4 *__restrict__ leaf, float3 pt, float3 *p, uint32_t *tri,
                                      uint32_t *feat, uint32_t *id) {
#pragma clang fp contract(off)
    const float4 va = leaf[0], vb = leaf[1], vc = leaf[2];
    *tri = __float_as_uint(va.w);
    *p = triangle_project(make_float3(va.x, va.y, va.z), make_float3(vb.x, vb.y, vb.z), make_float3(vc.x, vc.y, vc.z),
                          pt, feat, id);
    const float dx = p->x - pt.x, dy = p->y - pt.y, dz = p->z - pt.z;
    return sqrtf(dx * dx + dy * dy + dz * dz);
}

// Distance of a point from the box of the triangle of `leaf`.
__device__ inline float leaf_box_distance(const float4 *__restrict__ leaf, float3 pt) {
    const float4 a = leaf[0], b = leaf[1], c = leaf[2];
    return box_distance(make_float4(fminf(fminf(a.x, b.x), c.x), fminf(fminf(a.y, b.y), c.y), fminf(fminf(a.z, b.z), c.z), 0.0f),
                        make_float4(fmaxf(fmaxf(a.x, b.x), c.x), fmaxf(fmaxf(a.y, b.y), c.y), fmaxf(fmaxf(a.z, b.z), c.z), 0.0f),
                        pt);
}

// TriMesh::project_local_point (trimesh.slang:111-154): the leaf of the closest
// triangle within max_dist by the stackless BVH walk (SLOSH_NONE: none; links point
// forward, checked on the host, so the walk ends), each lane for its own point. With `cull`,
// a leaf whose box (grown by 1 % on the host, far above rounding) is farther than the best
// so far is skipped, which the reference tests all the same: no triangle but a degenerate
// one can win from there.
__device__ inline uint32_t trimesh_walk(const float4 *__restrict__ node, const float4 *__restrict__ leaf,
                                        uint32_t nodes, float3 pt, float max_dist, bool cull) {
    float best = max_dist;
    uint32_t best_leaf = SLOSH_NONE;
    for (uint32_t at = 0u; at < nodes;) {
        const float4 mn = node[2u * at], mx = node[2u * at + 1u];
        const uint32_t entry = __float_as_uint(mn.w), exit_ = __float_as_uint(mx.w);
        const float dbox = box_distance(mn, mx, pt);
        if (entry != SLOSH_NONE) {
            at = dbox < best ? entry : exit_;
            continue;
        }
        if (!cull || dbox <= best) {
            float3 p;
            uint32_t tri, feat, id;
            const float dist = leaf_distance(leaf + 3u * (size_t)at, pt, &p, &tri, &feat, &id);
            if (dist <= best) {
                best = dist;
                best_leaf = at;
            }
        }
        at = exit_;
    }
    return best_leaf;
}

// The projection on leaf `lf` of trimesh collider `i`, and TriMesh::pseudo_normal
// (trimesh.slang:83-109) of the feature it lies on, which tells inside from outside.
__device__ inline void trimesh_contact(const Colliders &cs, uint32_t i, uint32_t lf, float3 pt, float3 *out,
                                       bool *inside) {
#pragma clang fp contract(off)
    const float4 a = cs.shapes[2 * i], b = cs.shapes[2 * i + 1];
    const uint32_t vroot = __float_as_uint(a.x), iroot = __float_as_uint(a.y), nodes = __float_as_uint(a.z);
    const uint32_t nvert = __float_as_uint(b.y);
    const uint32_t *tri_idx = cs.mesh_idx + iroot + 3u * nodes;
    const float4 *verts = cs.mesh_vtx + vroot + 2u * nodes;
    uint32_t tri, feat, id;
    leaf_distance(cs.mesh_leaves + 3u * (size_t)(cs.mesh_base[i] + lf), pt, out, &tri, &feat, &id);
    float3 pn;
    const uint32_t *tv = tri_idx + 3u * tri;
    if (feat == 0u) {
        const float4 q = verts[tv[id] + nvert];
        pn = make_float3(q.x, q.y, q.z);
    } else if (feat == 1u) {
        const float4 q = verts[2u * nvert + 3u * tri + id];
        pn = make_float3(q.x, q.y, q.z);
    } else {
        const float4 va = verts[tv[0]], vb = verts[tv[1]], vc = verts[tv[2]];
        pn = cross3f(make_float3(vb.x - va.x, vb.y - va.y, vb.z - va.z),
                     make_float3(vc.x - va.x, vc.y - va.y, vc.z - va.z));
    }
    *inside = pn.x * (pt.x - out->x) + pn.y * (pt.y - out->y) + pn.z * (pt.z - out->z) <= 0.0f;
}

// The closest triangles of a block's 64 nodes by a workgroup of MESH_WAVES waves,
// for every trimesh collider: the leaves near the block are collected, of a small mesh
// from all its nodes at once, else by one wave, a level of the BVH at a time; then each
// wave tests its share of them for all nodes (lane = node), culled by the closest that
// any wave has found, and the closest wins by an LDS minimum over (distance, leaf).
//
// The walk (trimesh_walk) defines the result. It finds the same point, but for rounding, if
// every triangle lies in the boxes above it (the host says which meshes are such; MESH_WALK:
// not) and it cannot miss the closest one: a triangle farther than its own box is surely
// met, as the boxes above are nearer still. One at its box's distance (it lies along an
// axis, say) may be left out when another point is as far, or when the reach is, by the
// strict comparison with the boxes: such nodes are walked after all.
//
// Bound by latency: a block is 64 nodes with ~50 triangles in reach, and one triangle
// test ~300 dependent instructions, so one wave per block left the chip idle. The
// grid update of 85k particles over an 874-triangle heightfield (429 blocks): walked
// per lane 110 us, shared by 8 waves 28 us (4 waves 37, 16 waves 48), with the leaves from
// all nodes at once 23 us, culled together and the undecided nodes walked 23.5 us. Over
// finer heightfields, walked per lane and now: 3698 triangles 180 -> 48 us, 15842 329 ->
// 127, 178802 (too many near a block: walked, eight nodes to a wave) 1213 -> 812; over a flat
// aligned floor of 2048, most of whose nodes are walked after all, 41 -> 37; a tree with
// short boxes over 3698 triangles 181 -> 125.
#define MESH_WAVES 8  // (each has eight of the 64 nodes where they are walked)
#define MESH_CAND 2048   // leaves near a block that the workgroup shares; more are walked
#define MESH_FRONT 2048  // nodes of a level near a block
struct MeshShared {
    uint32_t cand[MESH_CAND];
    uint32_t front[2][MESH_FRONT];
    uint32_t n_cand;  // above MESH_CAND: more than fit
    unsigned long long key[SLOSH_MAX_COLLIDERS][NODES_PER_BLOCK];  // all ones: none in reach
    float point[3][NODES_PER_BLOCK];  // on the closest
    uint32_t tie[NODES_PER_BLOCK];    // least distance that the walk has to decide (float bits)
};

// MeshShared::key: the distance (float bits), the leaf (the later one first, as the walk
// decides ties).
__device__ inline unsigned long long mesh_key(float dist, uint32_t leaf) {
    return ((unsigned long long)__float_as_uint(dist) << 32) | ~leaf;
}
__device__ inline uint32_t key_leaf(unsigned long long key) { return ~(uint32_t)key; }
__device__ inline float key_distance(unsigned long long key) { return __uint_as_float((uint32_t)(key >> 32)); }

// Appends `v` of the lanes in `on` to list[0, *n) (wave-uniform *n); false if it does not fit.
__device__ inline bool push(uint32_t *list, uint32_t cap, uint32_t *n, bool on, uint32_t v) {
    const uint64_t m = __ballot(on);
    const uint32_t at = *n + (uint32_t)__popcll(m & lanemask_lt());
    if (on && at < cap) list[at] = v;
    *n += (uint32_t)__popcll(m);
    return *n <= cap;
}

// Leaves of trimesh `node` whose boxes come within `reach` of the box c +- e, into
// S.cand; by one wave.
__device__ inline void mesh_candidates(MeshShared &S, const float4 *__restrict__ node, float3 c, float3 e,
                                       float reach) {
    const uint32_t lane = lane_id();
    uint32_t n_cand = 0u, nf = 1u, cur = 0u;
    bool fits = true;
    if (lane == 0) S.front[0][0] = 0u;
    while (nf > 0u && fits) {
        uint32_t next = 0u;
        for (uint32_t b = 0; b < nf && fits; b += 64u) {
            __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const bool have = b + lane < nf;
            const uint32_t k = have ? S.front[cur][b + lane] : 0u;
            const float4 mn = node[2u * k], mx = node[2u * k + 1u];
            const float gx = fmaxf(fmaxf(mn.x - (c.x + e.x), (c.x - e.x) - mx.x), 0.0f);
            const float gy = fmaxf(fmaxf(mn.y - (c.y + e.y), (c.y - e.y) - mx.y), 0.0f);
            const float gz = fmaxf(fmaxf(mn.z - (c.z + e.z), (c.z - e.z) - mx.z), 0.0f);
            const bool near = have && gx * gx + gy * gy + gz * gz <= reach * reach;
            const uint32_t entry = __float_as_uint(mn.w), end = __float_as_uint(mx.w);
            fits = push(S.cand, MESH_CAND, &n_cand, near && entry == SLOSH_NONE, k);
            // The children: the entry, then each child's exit up to this node's.
            uint32_t ch = near && entry != SLOSH_NONE ? entry : end;
            while (fits && __ballot(ch != end)) {
                const bool on = ch != end;
                fits = push(S.front[cur ^ 1u], MESH_FRONT, &next, on, ch);
                if (on) ch = __float_as_uint(node[2u * ch + 1u].w);
            }
        }
        cur ^= 1u;
        nf = next;
    }
    if (lane == 0) S.n_cand = fits ? n_cand : SLOSH_NONE;
}

// The same by the whole workgroup from all of a small mesh's nodes at once, without the
// levels' chain of loads.
__device__ inline void mesh_candidates_flat(MeshShared &S, const float4 *__restrict__ node, uint32_t count, float3 c,
                                            float3 e, float reach) {
    for (uint32_t k = threadIdx.x; k < count; k += 64u * MESH_WAVES) {
        const float4 mn = node[2u * k], mx = node[2u * k + 1u];
        const float gx = fmaxf(fmaxf(mn.x - (c.x + e.x), (c.x - e.x) - mx.x), 0.0f);
        const float gy = fmaxf(fmaxf(mn.y - (c.y + e.y), (c.y - e.y) - mx.y), 0.0f);
        const float gz = fmaxf(fmaxf(mn.z - (c.z + e.z), (c.z - e.z) - mx.z), 0.0f);
        if (__float_as_uint(mn.w) == SLOSH_NONE && gx * gx + gy * gy + gz * gz <= reach * reach) {
            const uint32_t at = atomicAdd(&S.n_cand, 1u);
            if (at < MESH_CAND) S.cand[at] = k;
        }
    }
}

struct NodeColl {
    float4 normal_id; // normal.xyz, w = collider id (u32 bits)
    float4 point_valid; // point.xyz, w = valid (u32 bits)
};

// collide(), collide.slang:87-154 (primitive shapes and trimeshes; polylines
// take no part, as in the reference).
// World-space box around the region where collider i can report a contact
// (the shape grown by `reach` along each axis, plus a margin far above the
// rounding of collide()'s transforms). A point outside it is outside the shape
// and farther than `reach` from its projection along some axis, so collide()
// takes nothing from the collider there and skips it. A trimesh's box is its
// BVH root box. Polylines (which collide() skips) and unknown shape types (whose projection is the
// point itself: never a contact) get an empty box. MESH: the launch carries the
// trimesh buffers (otherwise no collider is a trimesh).
template <bool MESH>
__device__ inline void collider_box(const Colliders &cs, uint32_t i, float reach, float4 *lo, float4 *hi) {
    const float4 a = cs.shapes[2 * i];
    const uint32_t ty = __float_as_uint(a.w);
    if (ty > 4u && !(MESH && ty == 6u)) {
        *lo = make_float4(1.0e30f, 1.0e30f, 1.0e30f, 0.0f);
        *hi = make_float4(-1.0e30f, -1.0e30f, -1.0e30f, 0.0f);
        return;
    }
    // The shape's local bounding box (centre, half extents).
    float3 c = make_float3(0.0f, 0.0f, 0.0f), e;
    if (ty == 1u) {
        e = make_float3(a.x, a.y, a.z);
    } else if (ty == 0u) {
        e = make_float3(a.x, a.x, a.x);
    } else if (ty == 2u) {
        const float4 b = cs.shapes[2 * i + 1];
        c = make_float3(0.5f * (a.x + b.x), 0.5f * (a.y + b.y), 0.5f * (a.z + b.z));
        e = make_float3(0.5f * fabsf(b.x - a.x) + b.w, 0.5f * fabsf(b.y - a.y) + b.w, 0.5f * fabsf(b.z - a.z) + b.w);
    } else if (MESH && ty == 6u) {
        // The BVH root's box (the first node's AABB).
        const uint32_t vroot = __float_as_uint(a.x);
        const float4 mn = cs.mesh_vtx[vroot], mx = cs.mesh_vtx[vroot + 1u];
        c = make_float3(0.5f * (mn.x + mx.x), 0.5f * (mn.y + mx.y), 0.5f * (mn.z + mx.z));
        e = make_float3(0.5f * (mx.x - mn.x), 0.5f * (mx.y - mn.y), 0.5f * (mx.z - mn.z));
    } else {
        e = make_float3(a.y, a.x, a.y);  // cone / cylinder: radius, half height (axis y), radius
    }
    const float4 rot = cs.poses[2 * i], ts = cs.poses[2 * i + 1];
    // World box of the rotated, scaled local box: centre transformed, half extents |R| e |scale|.
    const float3 cw = sim_mul_pt(rot, ts, c);
    const float3 cx = quat_rotate(rot, make_float3(1.0f, 0.0f, 0.0f));
    const float3 cy = quat_rotate(rot, make_float3(0.0f, 1.0f, 0.0f));
    const float3 cz = quat_rotate(rot, make_float3(0.0f, 0.0f, 1.0f));
    const float sc = fabsf(ts.w);
    const float3 ext = make_float3((fabsf(cx.x) * e.x + fabsf(cy.x) * e.y + fabsf(cz.x) * e.z) * sc,
                                   (fabsf(cx.y) * e.x + fabsf(cy.y) * e.y + fabsf(cz.y) * e.z) * sc,
                                   (fabsf(cx.z) * e.x + fabsf(cy.z) * e.y + fabsf(cz.z) * e.z) * sc);
    const float size = fmaxf(fmaxf(ext.x, ext.y), ext.z) + fmaxf(fmaxf(fabsf(cw.x), fabsf(cw.y)), fabsf(cw.z));
    const float m = reach * 1.01f + 1.0e-4f * size;
    *lo = make_float4(cw.x - ext.x - m, cw.y - ext.y - m, cw.z - ext.z - m, 0.0f);
    *hi = make_float4(cw.x + ext.x + m, cw.y + ext.y + m, cw.z + ext.z + m, 0.0f);
}

// `box`: collider_box of each collider (reach 1.5 h). `keys`: per trimesh collider the
// point's closest leaf (MeshShared::key at the point's node).
template <bool MESH>
__device__ inline NodeColl collide(const Colliders &cs, const float4 *box, float h, float3 point,
                                   const unsigned long long (*keys)[NODES_PER_BLOCK], uint32_t lane) {
#pragma clang fp contract(off)
    NodeColl c;
    c.normal_id = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(0u));
    c.point_valid = make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(0u));
    float dist_cap = h * 1.5f;
    float best = 1.0e10f;
    for (uint32_t i = 0; i < cs.count; i++) {
        const float4 lo = box[2 * i], hi = box[2 * i + 1];
        if (point.x < lo.x || point.x > hi.x || point.y < lo.y || point.y > hi.y || point.z < lo.z || point.z > hi.z)
            continue;
        float4 a = cs.shapes[2 * i];
        uint32_t ty = __float_as_uint(a.w);
        if (ty == 5u) continue;
        float4 rot = cs.poses[2 * i], ts = cs.poses[2 * i + 1];
        float3 proj;
        bool inside = false;
        if (MESH && ty == 6u) {
            // collide.slang:120-130: only a triangle within dist_cap counts.
            const unsigned long long key = keys[i][lane];
            if (key == ~0ull) continue;
            float3 lproj;
            trimesh_contact(cs, i, key_leaf(key), sim_inv_mul_pt(rot, ts, point), &lproj, &inside);
            proj = sim_mul_pt(rot, ts, lproj);
        } else if (ty <= 4u) {
            float3 lp = sim_inv_mul_pt(rot, ts, point);
            float3 lproj;
            if (ty == 1u) {
                inside = cuboid_project_boundary(make_float3(a.x, a.y, a.z), lp, &lproj);
            } else if (ty == 0u) {
                inside = ball_project_boundary(a.x, lp, &lproj);
            } else if (ty == 2u) {
                const float4 b = cs.shapes[2 * i + 1];
                inside = capsule_project_boundary(make_float3(a.x, a.y, a.z), make_float3(b.x, b.y, b.z), b.w, lp,
                                                  &lproj);
            } else if (ty == 3u) {
                inside = cone_project_boundary(a.x, a.y, lp, &lproj);
            } else {
                inside = cylinder_project_boundary(a.x, a.y, lp, &lproj);
            }
            proj = sim_mul_pt(rot, ts, lproj);
        } else {
            proj = point; // shape.slang:200
        }
        float3 d = make_float3(proj.x - point.x, proj.y - point.y, proj.z - point.z);
        if (inside || (fabsf(d.x) <= dist_cap && fabsf(d.y) <= dist_cap && fabsf(d.z) <= dist_cap)) {
            float sign = inside ? -1.0f : 1.0f;
            float dist = sqrtf(d.x * d.x + d.y * d.y + d.z * d.z);
            if (sign * dist < best && dist != 0.0f) {
                float k = dist * -sign;
                c.normal_id = make_float4(d.x / k, d.y / k, d.z / k, __uint_as_float(i));
                c.point_valid = make_float4(proj.x, proj.y, proj.z, __uint_as_float(1u));
                best = dist;
            }
        }
    }
    return c;
}

// BoundaryCondition::project_velocity, boundary_condition.slang:31-89
__device__ inline float3 project_velocity(uint2 bc, float3 v, float3 n, float dist, float dt) {
    uint32_t ty = bc.x;
    float friction = __uint_as_float(bc.y);
    if (ty == 0u) {
        if (dist <= 0.0f) return make_float3(0.0f, 0.0f, 0.0f);
        return v;
    }
    if (ty == 1u) {
        if (dist <= 0.0f) {
            float nv = v.x * n.x + v.y * n.y + v.z * n.z;
            return make_float3(v.x - n.x * nv, v.y - n.y * nv, v.z - n.z * nv);
        }
        return v;
    }
    if (ty == 2u || ty == 3u) {
        float nv = v.x * n.x + v.y * n.y + v.z * n.z;
        if (nv < 0.0f) {
            if (dist <= 0.0f) {
                float3 tv = make_float3(v.x - n.x * nv, v.y - n.y * nv, v.z - n.z * nv);
                float tl = sqrtf(tv.x * tv.x + tv.y * tv.y + tv.z * tv.z);
                float3 dir = make_float3(0.0f, 0.0f, 0.0f);
                if (tl > 1.0e-8f) dir = make_float3(tv.x / tl, tv.y / tl, tv.z / tl);
                float m = fmaxf(0.0f, tl + friction * nv);
                return make_float3(dir.x * m, dir.y * m, dir.z * m);
            } else if (-nv * dt > dist) {
                float k = dist / dt + nv;
                return make_float3(v.x - k * n.x, v.y - k * n.y, v.z - k * n.z);
            }
        }
        return v;
    }
    return v;
}

// ---------------------------------------------------------------------------
// Particle state views.

struct PBuf {
    float4 *pos;    // xyz, w = (scene << 1 | enabled) bits
    float4 *vm;     // velocity xyz, mass
    float *C;       // [9][pcap]
    float *F;       // [9][pcap]
    float *vgd;     // [pcap]
    uint32_t *ids;  // original index
    float *dps;     // [3][pcap] Drucker-Prager state (sand only)
};

struct PStatic {
    const float4 *prop;  // by original id: (V0, damping, fixed bits, radius)
    const float4 *model; // by original id: (tag bits, lambda, mu, cfl) of the elastic part
    const float4 *dp0;   // by original id: (h0, h1, h2, h3)
    const float4 *dp1;   // by original id: (lambda, mu, 0, 0) of the plastic part
    const float4 *scene_rec;  // batched, one record per scene: prop, model, dp0, dp1 per scene id
};

// A particle's static records: the single record, its scene's record, or its own
// (by original id).
__device__ inline void static_records(const StepParams &P, const PStatic &st, uint32_t oid, uint32_t scene,
                                      float4 *prop, float4 *model) {
    if (P.uniform) {
        *prop = P.u_prop;
        *model = P.u_model;
    } else if (P.scene_uniform) {
        *prop = st.scene_rec[4 * (size_t)scene];
        *model = st.scene_rec[4 * (size_t)scene + 1];
    } else {
        *prop = st.prop[oid];
        *model = st.model[oid];
    }
}

__device__ inline void plastic_records(const StepParams &P, const PStatic &st, uint32_t oid, uint32_t scene,
                                       float4 *dp0, float4 *dp1) {
    if (P.uniform) {
        *dp0 = P.u_dp0;
        *dp1 = P.u_dp1;
    } else if (P.scene_uniform) {
        *dp0 = st.scene_rec[4 * (size_t)scene + 2];
        *dp1 = st.scene_rec[4 * (size_t)scene + 3];
    } else {
        *dp0 = st.dp0[oid];
        *dp1 = st.dp1[oid];
    }
}

// G2P of one particle from the 6x6x6 LDS halo (g2p.slang:150-265):
// v = sum w v_i, C = (4/h^2) sum w v_i dpt_i^T, vel_grad_det = (4/h^2) sum w v_i . dpt_i.
// With dpt_i = ref + s_i h (s_i in {0,1,2}^3 the node's stencil shift), the sums
// are formed from V = sum w v_i and S_a = sum w s_i,a v_i (a = x, y, z):
// sum w v_i dpt_i,a = V ref_a + h S_a.
// `at`: the particle's stencil; lc: its associated cell's place in the block.
__device__ inline void g2p_particle(const float4 *__restrict__ sh, float h, float inv_d, const Stencil &at,
                                    const uint32_t *lc, bool enabled, float3 *vel, float *vg, float *vgd_out) {
    float V[3] = {0.0f, 0.0f, 0.0f}, S[3][3] = {{0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f}};
    float ref[3] = {0.0f, 0.0f, 0.0f};
    if (enabled) {
        float w[3][3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            ref[i] = at.ref[i];
            k_eval_all(at.f[i], w[i]);
        }
        const uint32_t packed = lc[0] + lc[1] * 6u + lc[2] * 36u;
        // V = sum_n w_n v_n and S[d] = sum_n s_d(n) w_n v_n (s_d = the node's stencil
        // offset 0..2 along d), with the separable weight w_n = wx wy wz summed
        // one axis at a time: rows along x first, then y within each z slab, then z.
        const float wx2 = 2.0f * w[0][2], wy2 = 2.0f * w[1][2], wz2 = 2.0f * w[2][2];
#pragma unroll
        for (int sz = 0; sz < 3; sz++) {
            float bz[3] = {0.0f, 0.0f, 0.0f}, myz[3] = {0.0f, 0.0f, 0.0f}, mxz[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int sy = 0; sy < 3; sy++) {
                const uint32_t base = packed + (uint32_t)sy * 6u + (uint32_t)sz * 36u;
                const float4 c0 = sh[base], c1 = sh[base + 1u], c2 = sh[base + 2u];
                const float r[3] = {w[0][0] * c0.x + w[0][1] * c1.x + w[0][2] * c2.x,
                                    w[0][0] * c0.y + w[0][1] * c1.y + w[0][2] * c2.y,
                                    w[0][0] * c0.z + w[0][1] * c1.z + w[0][2] * c2.z};
                const float mx[3] = {w[0][1] * c1.x + wx2 * c2.x, w[0][1] * c1.y + wx2 * c2.y,
                                     w[0][1] * c1.z + wx2 * c2.z};
                const float wy = w[1][sy];
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    bz[c] += wy * r[c];
                    mxz[c] += wy * mx[c];
                    if (sy == 1) myz[c] += wy * r[c];
                    if (sy == 2) myz[c] += wy2 * r[c];
                }
            }
            const float wz = w[2][sz];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                V[c] += wz * bz[c];
                S[0][c] += wz * mxz[c];
                S[1][c] += wz * myz[c];
                if (sz == 1) S[2][c] += wz * bz[c];
                if (sz == 2) S[2][c] += wz2 * bz[c];
            }
        }
    }
    *vel = make_float3(V[0], V[1], V[2]);
    float vgd = 0.0f;
#pragma unroll
    for (int r = 0; r < 3; r++) {
#pragma unroll
        for (int c = 0; c < 3; c++) vg[r * 3 + c] = inv_d * (V[c] * ref[r] + h * S[r][c]);
        vgd += V[r] * ref[r] + h * S[r][r];
    }
    *vgd_out = inv_d * vgd;
}

// particle_update.slang:32-160 for one particle, in three parts. No multiply-add
// contraction here or in the stress helpers: F - I and mu (F F^T - I) are small
// differences of O(1) values, so each rounding step shows in them; unfused
// products and sums round like the shader source's separate operations.

// The first part: velocity clamp, damping and fixing, the new position, F += F
// (dt aff) (`aff` is the velocity gradient, zeroed for a fixed particle).
__device__ inline void advance_particle(const StepParams &P, float3 pos, float3 &v, float *aff, float *F, float4 prop,
                                        float3 *np) {
#pragma clang fp contract(off)
    const float dt = P.dt, h = P.h;
    float vl = sqrtf(v.x * v.x + v.y * v.y + v.z * v.z);
    if (vl > P.h_dt) {
        float l2 = sqrtf(v.x * v.x + v.y * v.y + v.z * v.z);
        v = make_float3(v.x / l2 * h / dt, v.y / l2 * h / dt, v.z / l2 * h / dt);
    }
    float damp = 1.0f + prop.y * dt;
    if (damp != 1.0f) v = make_float3(v.x / damp, v.y / damp, v.z / damp);
    bool fixed = __float_as_uint(prop.z) != 0u;
    if (fixed) v = make_float3(0.0f, 0.0f, 0.0f);
    *np = make_float3(pos.x + v.x * dt, pos.y + v.y * dt, pos.z + v.z * dt);
    // F += mul(F, affine * dt)
    float adt[9], fa[9];
#pragma unroll
    for (int k = 0; k < 9; k++) adt[k] = aff[k] * dt;
    mul3(F, adt, fa);
#pragma unroll
    for (int k = 0; k < 9; k++) F[k] = F[k] + fa[k];
    if (fixed) {
#pragma unroll
        for (int k = 0; k < 9; k++) aff[k] = 0.0f;
    }
}

// The second part, DefaultParticleModel::update (default.slang:51-92): the plastic
// projection of F and the stress. MODELS is the set of material tags the kernel
// instance handles (bit t = tag t), so scenes without SVD-based models do not
// carry that code's register footprint.
template <uint32_t MODELS, bool F64>
__device__ inline void material_update(const StepParams &P, float *F, float4 model, const PStatic &st, uint32_t oid,
                                       uint32_t scene, float *dps, float *stress) {
    // A wave of several materials runs each step once, for the lanes of all the tags
    // that take it.
    const uint32_t tag = __float_as_uint(model.x);
    if (((MODELS & 4u) && tag == 2u) || ((MODELS & 8u) && tag == 3u)) {
        float4 hp, pl;
        plastic_records(P, st, oid, scene, &hp, &pl);
        if (F64) dp_project_f64(dps, hp, pl.x, pl.y, F);
        else dp_project(dps, hp, pl.x, pl.y, F);
    }
    if (((MODELS & 1u) && tag == 0u) || ((MODELS & 4u) && tag == 2u)) {
        if (F64) fc_stress_f64(model.y, model.z, F, stress);
        else fc_stress(model.y, model.z, F, stress);
    } else if (((MODELS & 2u) && tag == 1u) || ((MODELS & 8u) && tag == 3u)) {
        nh_stress(model.y, model.z, F, stress);
    } else {
#pragma unroll
        for (int k = 0; k < 9; k++) stress[k] = 0.0f;
    }
}

// The third part: whether the particle stays enabled (a finite position and
// det F > 0), and its APIC affine matrix (from the velocity gradient, in `aff`);
// a particle that is disabled gets zeros and F = I.
__device__ inline bool stays_enabled(float3 np, const float *F) {
    return np.x == np.x && np.y == np.y && np.z == np.z && det3(F) > 0.0f;
}

__device__ inline void finish_particle(const StepParams &P, bool ok, float mass, float init_volume, const float *stress,
                                       float *aff, float *F) {
#pragma clang fp contract(off)
    const float sk = init_volume * P.inv_d * P.dt;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        if (ok) {
            aff[k] = aff[k] * mass - stress[k] * sk;
        } else {
            F[k] = (k == 0 || k == 4 || k == 8) ? 1.0f : 0.0f;
            aff[k] = 0.0f;
        }
    }
}

// ---------------------------------------------------------------------------
// A block's particles ("members").

// In the steady state a block's members are the particles of its range in the
// previous substep's storage that are still in the block ("candidates": the
// range is read whole and filtered by block; prev_stay of them pass) and the
// movers listed for it (MOVER_CAP list slots per block, the rest in the
// overflow list). After a full sort they are the sorted list
// perm[blk_start, blk_start + blk_cnt).
struct Members {
    uint32_t fast;
    const uint32_t *blist;                   // block list (header ids = table slots)
    const uint4 *bin;                        // per block: its previous-table block's range (start, count) and
                                             // stayers, the movers it received
    const uint32_t *mlist;                   // the first MOVER_CAP of them
    const uint32_t *ovf_slot, *ovf_hid;      // the others
    const uint32_t *perm, *blk_start, *blk_cnt;  // the full sort's result
    const uint32_t *counters;                // CTR_NUM_BLOCKS, CTR_OVERFLOW of this substep
};

// What P2G of a steady-state substep finds and leaves for the kernels after it: the
// regional block lists, what each block receives (movers; slot, start and count in the
// previous table), the previous table's keys and stayers; the flat block list, each
// block's range (Members::bin) and neighbour table.
struct SortInputs {
    const uint2 *rlist;
    const uint4 *arrive;
    const uint32_t *rcnt, *prev_keys, *prev_stay;
    uint32_t *blist, *num_blocks, *nbr, *blk_cnt;
    uint4 *bin;
    // Per region (slot >> rshift) the sums of its blocks' particles (high word) and G2P
    // items (low word), and each block's place in them.
    unsigned long long *rsum;
    uint2 *rel;
    uint32_t rshift;
};

struct BlockRange {
    uint32_t cand_lo, cand_n;  // candidates: storage slots [cand_lo, cand_lo + cand_n)
    const uint32_t *list;      // then the members list[0, list_n)
    uint32_t list_n;
    uint32_t total;            // members, overflow movers included
    bool overflow;             // some of the block's movers are in the overflow list
};

// FAST (a template parameter, so that each kernel instance loads only the
// buffers of its mode): the steady state's stayer ranges and mover lists.
__device__ inline BlockRange steady_range(const Members &M, uint32_t hid, uint4 in) {
    const uint32_t mc = in.w;
    BlockRange r;
    r.cand_lo = in.x;
    r.cand_n = in.y;
    r.list = M.mlist + (size_t)hid * MOVER_CAP;
    r.list_n = mc < MOVER_CAP ? mc : MOVER_CAP;
    r.total = in.z + mc;
    r.overflow = mc > MOVER_CAP;
    return r;
}

template <bool FAST>
__device__ inline BlockRange block_range(const Members &M, uint32_t hid) {
    if constexpr (FAST) return steady_range(M, hid, M.bin[hid]);
    BlockRange r;
    r.cand_lo = 0u;
    r.cand_n = 0u;
    r.list = M.perm + M.blk_start[hid];
    r.list_n = M.blk_cnt[hid];
    r.total = r.list_n;
    r.overflow = false;
    return r;
}

// G2P items of a block: 64 entries each.
__device__ inline uint32_t item_count(const BlockRange &r) { return r.total ? (r.cand_n + r.list_n + 63u) >> 6 : 0u; }

// Storage slot of entry m of a block's sequence (candidates, then list members).
__device__ inline uint32_t entry_slot(const BlockRange &r, uint32_t m) {
    return m < r.cand_n ? r.cand_lo + m : r.list[m - r.cand_n];
}

// ---------------------------------------------------------------------------
// Kernels.

// P2G for one block per workgroup of 3 SUB waves.
// Phase 1 (per chunk of up to P2G_CHUNK members of the block): each thread
// loads one particle (stayers are contiguous in storage) and stages in LDS what
// every node of its stencil shares: mass, the APIC momentum at the stencil's
// first node A0 = m v + C^T (x_0 - x_p), the particle's offset f from that node
// in cells (the kernel weights follow from it in a few operations, cheaper than
// staging them: LDS per particle bounds how many workgroups share a CU), and C.
// The chunk is grouped by associated cell in LDS (a rank per particle from an
// LDS counter per cell, a scan of the 64 counts, a list of staging indices).
// Phase 2: lane = associated cell of the block, wave = z offset kz of the
// stencil (and which of every SUB members of the cell); each lane accumulates, over the particles of its cell in the chunk,
// the contributions w_n (A0 + C^T (n h)) to the 9 nodes n = (kx, ky, kz) in 36
// registers.
// Phase 3: each wave sums its registers into its own slab tile (z planes kz to
// kz + 3 of the 6x6x6 tile, in the LDS of the staging), in 9 rounds in which its
// 64 lanes touch 64 distinct nodes (plain read-modify-write; no LDS or global
// atomics on floats), all three waves at once; then each node of the tile is
// the sum of the slabs that cover it, in wave order, written straight to HBM.
// Each cell's summation order follows the order its particles were grouped in.
// Cells hold ~8 particles, so lanes read particles ~8 apart: one padding element
// every 16 spreads 16 consecutive cells' first particles over the 16 LDS bank
// groups of 16-byte elements.
__device__ inline uint32_t p2g_slot(uint32_t q) { return q + (q >> 4); }

// LDS element of node (x, y, z) of a P2G slab tile (z = 0..3), 16-byte elements.
// Within a z plane, x < 4 maps to x + 4 y (0..23) and x >= 4 to x + 4 y + 24
// (28..49), one to one;
// over any 4x4 patch of a plane (the 16 lanes of one merge access, at offsets
// 0..2 in x and y) the element index mod 16, its LDS bank group, takes 16
// different values (the patch's columns differ mod 4, and each column's 4 rows
// cover the residues of that class).
#define P2G_SLAB_LDS 200
__device__ inline uint32_t p2g_tile_lds(uint32_t x, uint32_t y, uint32_t z) {
    return x + 4u * y + (x >= 4u ? 24u : 0u) + 50u * z;
}

// 35,088 bytes at 512 particles per chunk: four workgroups (12 waves) fit in a
// CU's 160 KiB of LDS, as many as the registers allow; 26,384 bytes at 384.
template <int P2G_CHUNK, int SUB>
struct P2GShared {
    static constexpr int LDS = P2G_CHUNK + P2G_CHUNK / 16;
    union {
        // (m, A0), (f, C0), (C1..C4), (C5..C8) per member, grouped by associated cell
        float4 sp4[4][LDS];
        // after the block's last chunk: each wave's sums over its slab (z planes kz..kz+3)
        float4 slab[3 * SUB][P2G_SLAB_LDS];
        uint32_t extra[192 * SUB];  // this block's overflow movers of one round: read by
                                    // p2g_chunk before it stages anything
    };
    uint32_t lcnt[64];
    uint32_t wsum[3 * SUB];
};
static_assert(sizeof(float4) * 3 * P2G_SLAB_LDS <= sizeof(P2GShared<192, 1>::sp4),
              "the slab tiles take no LDS beyond the staging of the smallest chunk");
static_assert(sizeof(P2GShared<512, 1>) <= 163840 / 4, "P2G at 512 per chunk must fit four workgroups per CU");

// Phase 1 and 2 for `kn` entries of the block's sequence; entry t's storage slot
// is slot_of(t). An entry is a member if its associated block is this block
// (candidates that moved to another block are skipped; every other entry is one
// by construction). Every thread of the workgroup calls it. `tot` (wave 0, lane
// = cell) accumulates the block's cell counts.
template <int P2G_CHUNK, int SUB, typename SlotOf>
__device__ inline void p2g_chunk(const StepParams &P, P2GShared<P2G_CHUNK, SUB> &S, uint32_t kn, SlotOf slot_of, const float4 *__restrict__ pos, const float4 *__restrict__ vm,
                                 const float *__restrict__ C, const float *__restrict__ fdt, uint32_t pcap,
                                 uint32_t block_key, float (&acc)[9][4], uint32_t &tot) {
    constexpr uint32_t T = 192 * SUB;
    constexpr int R = (P2G_CHUNK + T - 1) / T;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t kz = SUB == 1 ? wave : wave % 3u, part = SUB == 1 ? 0u : wave / 3u;
    const float h = P.h;
    const float kzh = (float)kz * h;
    // The slab's z weight is one piece of the quadratic B-spline of the offset f,
    // the same for the whole wave: wz = a (f - b)^2 + c (no divergent branch).
    const uint32_t kzu = __builtin_amdgcn_readfirstlane(kz);
    const float wza = kzu == 1u ? -1.0f : 0.5f;
    const float wzb = kzu == 0u ? 1.5f : (kzu == 1u ? 1.0f : 0.5f);
    const float wzc = kzu == 1u ? 0.75f : 0.0f;
    __syncthreads();  // the previous chunk's readers are done; the cell counters are clear
    // All of this thread's loads are issued before any is consumed.
    uint32_t pp[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t t = threadIdx.x + T * r;
        pp[r] = t < kn ? slot_of(t) : SLOSH_NONE;
    }
    float4 ps[R], vv[R];
    float cc[R][9];
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (pp[r] != SLOSH_NONE) {
            ps[r] = pos[pp[r]];
            vv[r] = vm[pp[r]];
#pragma unroll
            for (int k = 0; k < 9; k++) cc[r][k] = C[(size_t)k * pcap + pp[r]];
        }
    }
    // Per member: the associated cell, a rank within it, and the staged terms.
    uint32_t cl[R], rk[R];
    float a0[R][3], fo[R][3];
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (pp[r] == SLOSH_NONE) continue;
        float mom[3] = {vv[r].x * vv[r].w, vv[r].y * vv[r].w, vv[r].z * vv[r].w};
        if (P.has_force) {
#pragma unroll
            for (int i = 0; i < 3; i++) mom[i] += fdt[(size_t)i * pcap + pp[r]];
        }
        // The associated cell: node 0 of the stencil sits at d0 = x_0 - x_p; its
        // block (floor of the cell / 4) and its place in that block.
        const Stencil at = stencil_of(h, ps[r].x, ps[r].y, ps[r].z);
        int blk[3];
        uint32_t lc[3];
        block_of_cell(at.cell, blk, lc);
        const float *d0 = at.ref;
#pragma unroll
        for (int i = 0; i < 3; i++) fo[r][i] = at.f[i];
        // A candidate that moved to another block is that block's member.
        if (pack_key(P.batched, __float_as_uint(ps[r].w) >> 1, blk[0], blk[1], blk[2]) != block_key) {
            pp[r] = SLOSH_NONE;
            continue;
        }
        const float *c = cc[r];
#pragma unroll
        for (int i = 0; i < 3; i++) a0[r][i] = mom[i] + (d0[0] * c[i] + d0[1] * c[3 + i] + d0[2] * c[6 + i]);
        cl[r] = lc[0] + 4u * lc[1] + 16u * lc[2];
        rk[r] = atomicAdd(&S.lcnt[cl[r]], 1u);
    }
    __syncthreads();
    // Every wave scans the 64 counts (lane = cell) and writes the same starts.
    const uint32_t cnt = S.lcnt[lane];
    const uint32_t cs = wave_inclusive_scan(cnt) - cnt;
    if (wave == 0) tot += cnt;
    // Each member's cell start from the lane of its cell (every wave holds all 64).
    uint32_t cstart[R];
#pragma unroll
    for (int r = 0; r < R; r++) cstart[r] = (uint32_t)__shfl((int)cs, pp[r] != SLOSH_NONE ? (int)cl[r] : 0);
    // Staging in cell order: a cell's members are consecutive.
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (pp[r] == SLOSH_NONE) continue;
        const uint32_t q = p2g_slot(cstart[r] + rk[r]);
        S.sp4[0][q] = make_float4(vv[r].w, a0[r][0], a0[r][1], a0[r][2]);
        S.sp4[1][q] = make_float4(fo[r][0], fo[r][1], fo[r][2], cc[r][0]);
        S.sp4[2][q] = make_float4(cc[r][1], cc[r][2], cc[r][3], cc[r][4]);
        S.sp4[3][q] = make_float4(cc[r][5], cc[r][6], cc[r][7], cc[r][8]);
    }
    __syncthreads();
    for (uint32_t j = cs + part; j < cs + cnt; j += SUB) {
        const uint32_t q = p2g_slot(j);
        const float4 s0 = S.sp4[0][q], s1 = S.sp4[1][q], s2 = S.sp4[2][q], s3 = S.sp4[3][q];
        const float m = s0.x;
        const float a0s[3] = {s0.y, s0.z, s0.w};
        const float tz = s1.z - wzb;
        const float wz = fmaf(wza * tz, tz, wzc);
        float wx[3], wy[3], wyz[3], az[3];
        const float c[9] = {s1.w, s2.x, s2.y, s2.z, s2.w, s3.x, s3.y, s3.z, s3.w};
        k_eval_all(s1.x, wx);
        k_eval_all(s1.y, wy);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            wyz[i] = wy[i] * wz;
            // A0 + C^T (0, 0, kz h): shared by the 9 nodes of the slab.
            az[i] = a0s[i] + kzh * c[6 + i];
        }
#pragma unroll
        for (int ky = 0; ky < 3; ky++) {
            float ay[3];
#pragma unroll
            for (int i = 0; i < 3; i++) ay[i] = ky == 0 ? az[i] : az[i] + (float)ky * h * c[3 + i];
#pragma unroll
            for (int kx = 0; kx < 3; kx++) {
                const int k = kx + 3 * ky;
                const float wgt = wx[kx] * wyz[ky];
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const float a = kx == 0 ? ay[i] : ay[i] + (float)kx * h * c[i];
                    acc[k][i] += a * wgt;
                }
                acc[k][3] += m * wgt;
            }
        }
    }
    __syncthreads();
    if (wave == 0) S.lcnt[lane] = 0u;
}

// Key and first slot of entry `lane` (see NBR_STRIDE) of a block's neighbour table.
__device__ inline uint32_t neighbour_key(const StepParams &P, uint32_t block_key, uint32_t lane, uint32_t *slot) {
    int bx, by, bz;
    uint32_t scene;
    unpack_key(P.batched, block_key, &bx, &by, &bz, &scene);
    const int d = lane == NBR_PREV ? 0 : (int)(lane & 7u) + 1, s = lane < NBR_MINUS ? 1 : -1;
    const uint32_t key = pack_key(P.batched, scene, bx + s * ((d >> 2) & 1), by + s * ((d >> 1) & 1), bz + s * (d & 1));
    *slot = hash_key(key) & (P.cap - 1u);
    return key;
}

// The neighbours' first probes: most lookups end there, and the load is in flight
// through the block's sums.
__device__ inline uint32_t probe_neighbours(const StepParams &P, const SortInputs &in, const uint32_t *__restrict__ keys,
                                            uint32_t block_key, uint32_t lane) {
    uint32_t slot, seen = 0u;
    neighbour_key(P, block_key, lane, &slot);
    if (lane < NBR_MINUS + 7u) seen = (lane == NBR_PREV ? in.prev_keys : keys)[slot];
    return seen;
}

// By P2G's first wave, of a steady-state block: the rest of the lookups, and what the
// kernels after it read.
__device__ inline void finish_block(const StepParams &P, const SortInputs &in, const uint32_t *__restrict__ keys,
                                    uint32_t hid, uint32_t block_key, uint32_t lane, uint4 range, uint32_t total,
                                    uint32_t seen) {
    uint32_t slot;
    const uint32_t key = neighbour_key(P, block_key, lane, &slot);
    if (lane < NBR_MINUS + 7u) {
        const uint32_t *table = lane == NBR_PREV ? in.prev_keys : keys;
        for (uint32_t k = 1; seen != key && seen != SLOSH_NONE && k < P.cap; k++) {
            slot = (slot + 1u) & (P.cap - 1u);
            seen = table[slot];
        }
        in.nbr[(size_t)hid * NBR_STRIDE + lane] = seen == key ? slot : SLOSH_NONE;
    }
    if (lane == 0u) {
        in.bin[hid] = range;
        in.blk_cnt[hid] = total;
    }
}

// One workgroup per block, a block's on the XCD that also updates its nodes and
// particles (xcd_item); SUB = 2 gives each cell's members to two sets of three waves. In
// the steady state it starts from the regional lists and the ranges the previous substep
// left. A block takes ~6 us from its first dependent load (list entry, range, member
// slots, particles) to its tile, so what counts with many blocks is how many are
// resident: 512 members per chunk hold four workgroups to a CU (35 KB of LDS, 128 VGPRs),
// 384 let in five (106 VGPRs): 1M particles 43 -> 39 us, 48 scenes 101 -> 88, 2.1M in 42k
// blocks 248 -> 206 (36, 77 and 200 by now; more waves per SIMD at 96 VGPRs gain nothing).
// Chunks of 256 or 192 take more rounds (by now: 1M 36, 42; 48 scenes 82, 79; 131k 15, 20),
// which only the sparse blocks of the 2.1M do not have (203, 186).
// While all blocks are resident at once, the longest one's latency counts instead: a
// block of 512 then goes in one chunk (131k particles: 14.2 us against 15.3), and with a
// CU for each, in six waves that halve its longest cells and its loads per thread (2k
// particles 11.8 -> 9.7 us, 33k 12.2 -> 10.4, 80k 12.6 -> 12.2; but 131k 14.2 -> 16.6,
// 2.1M 248 -> 437). The count of blocks is not known to the host; scenes have one (with
// the empty neighbours) per 150 to 300 particles. Sprays of fewer have many more blocks and
// would do better with three waves: the substep of 90k particles, 6 to a block 101 us
// instead of 119, 2 to a block 244 instead of 312.
#define P2G_SUB_N 98304u    // two sets of waves up to here
#define P2G_WIDE_N 262144u  // chunks of 512 up to here

// (read through late_args: 14 to 26 scalar registers spilled otherwise; 48 scenes 87 -> 84.5
// us, 2.1M 206 -> 201)
struct P2gArgs {
    StepParams P;
    const float4 *pos, *vm;
    const float *C, *fdt;
    uint32_t pcap;
    Members M;
    SortInputs in;
    const uint32_t *keys;
    float4 *tiles;
    uint32_t *cell_cnt;
};

template <int P2G_CHUNK, bool FAST, int SUB>
__global__ __launch_bounds__(192 * SUB, SUB == 1 && P2G_CHUNK <= 384 ? 4 : 1) void k_p2g(P2gArgs args) {
    __shared__ P2GShared<P2G_CHUNK, SUB> S;
    constexpr uint32_t T = 192 * SUB;
    const uint32_t n_ovf = args.M.counters[CTR_OVERFLOW];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const int lx = lane & 3, ly = (lane >> 2) & 3, lz = lane >> 4;
    uint32_t B, upto = 0u;  // blocks; FAST: those of the regions up to the lane's
    if constexpr (FAST) {
        upto = wave_inclusive_scan(args.in.rcnt[lane * RCNT_STRIDE]);
        B = __builtin_amdgcn_readlane(upto, 63);
        if (blockIdx.x == 0u && threadIdx.x == 0u) *args.in.num_blocks = B;
    } else {
        B = args.M.counters[CTR_NUM_BLOCKS];
    }
    if (threadIdx.x < 64) S.lcnt[threadIdx.x] = 0u;
    for (uint32_t j = blockIdx.x >> 3;; j += gridDim.x >> 3) {
        const uint32_t k = xcd_item(blockIdx.x & 7u, j, B);
        if (k >= B) break;
        const P2gArgs &A = late_args<P2gArgs>();
        const StepParams &P = A.P;
        const Members &M = A.M;
        const SortInputs &in = A.in;
        const uint32_t *keys = A.keys;
        uint32_t hid, block_key;
        BlockRange br;
        uint4 range;
        uint32_t seen = 0u;
        if constexpr (FAST) {
            const uint32_t r = (uint32_t)__popcll(__ballot(upto <= k));
            const uint32_t before = r ? __builtin_amdgcn_readlane(upto, r - 1u) : 0u;
            const uint2 e = in.rlist[(r << in.rshift) + (k - before)];
            hid = __builtin_amdgcn_readfirstlane(e.x);
            block_key = __builtin_amdgcn_readfirstlane(e.y);
            const uint4 a = in.arrive[hid];
            const uint32_t prev = __builtin_amdgcn_readfirstlane(a.y);
            range = make_uint4(0u, 0u, 0u, __builtin_amdgcn_readfirstlane(a.x));
            if (prev != SLOSH_NONE) {
                range.x = __builtin_amdgcn_readfirstlane(a.z);
                range.y = __builtin_amdgcn_readfirstlane(a.w);
                range.z = in.prev_stay[prev];
            }
            br = steady_range(M, hid, range);
            if (wave == 0u) seen = probe_neighbours(P, in, keys, block_key, lane);
            if (threadIdx.x == 0u) in.blist[k] = hid;
        } else {
            hid = M.blist[k];
            block_key = keys[hid];
            br = block_range<false>(M, hid);
        }
        // A block without particles (a "+1" neighbour only) has an all-zero tile:
        // nothing is written and the grid update skips it. (The stayers are waited for
        // only below: a block that all its particles left writes a zero tile.)
        const uint32_t n_main = br.cand_n + br.list_n;
        if (n_main == 0u) {
            if (wave == 0u) {
                A.cell_cnt[(size_t)hid * NODES_PER_BLOCK + lane] = 0u;
                if constexpr (FAST) finish_block(P, in, keys, hid, block_key, lane, range, br.total, seen);
            }
            continue;
        }
        float acc[9][4];
#pragma unroll
        for (int q = 0; q < 9; q++) acc[q][0] = acc[q][1] = acc[q][2] = acc[q][3] = 0.0f;
        uint32_t tot = 0u;
        for (uint32_t chunk = 0; chunk < n_main; chunk += P2G_CHUNK) {
            const uint32_t kn = n_main - chunk < (uint32_t)P2G_CHUNK ? n_main - chunk : (uint32_t)P2G_CHUNK;
            p2g_chunk<P2G_CHUNK, SUB>(P, S, kn, [&](uint32_t t) { return entry_slot(br, chunk + t); }, A.pos, A.vm,
                                      A.C, A.fdt, A.pcap, block_key, acc, tot);
        }
        if (br.overflow) {
            // This block's movers beyond its list: picked out of the overflow list,
            // one round of T entries at a time.
            for (uint32_t ob = 0; ob < n_ovf; ob += T) {
                const uint32_t i = ob + threadIdx.x;
                const bool mine = i < n_ovf && M.ovf_hid[i] == hid;
                const uint64_t mm = __ballot(mine);
                __syncthreads();  // the previous round's readers of `extra` are done
                if (lane == 0) S.wsum[wave] = (uint32_t)__popcll(mm);
                __syncthreads();
                uint32_t before = 0u, kn = 0u;
#pragma unroll
                for (uint32_t w = 0; w < 3u * SUB; w++) {
                    before += w < wave ? S.wsum[w] : 0u;
                    kn += S.wsum[w];
                }
                if (mine) S.extra[before + (uint32_t)__popcll(mm & lanemask_lt())] = M.ovf_slot[i];
                if (kn > 0)
                    p2g_chunk<P2G_CHUNK, SUB>(P, S, kn, [&](uint32_t t) { return S.extra[t]; }, A.pos, A.vm, A.C, A.fdt,
                                              A.pcap, block_key, acc, tot);
            }
        }
        const P2gArgs &E = late_args<P2gArgs>();
        // The block's place in its region's storage and items (stored below).
        unsigned long long rel = 0ull;
        if (threadIdx.x == 0u)
            rel = atomicAdd(&E.in.rsum[(hid >> E.in.rshift) * RSUM_STRIDE], ((unsigned long long)br.total << 32) | item_count(br));
        // Each wave adds its registers into its own slab tile (sharing the staging's
        // LDS), in 9 rounds in which its 64 lanes touch 64 distinct nodes; then each
        // node is the sum of the slabs that cover it, in wave order.
        __syncthreads();  // the staging's readers are done
        float4 *slab = S.slab[wave];
        for (uint32_t j = lane; j < P2G_SLAB_LDS; j += 64) slab[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        __asm__ volatile("" ::: "memory");
#pragma unroll
        for (int ky = 0; ky < 3; ky++)
#pragma unroll
            for (int kx = 0; kx < 3; kx++) {
                const int q = kx + 3 * ky;
                const uint32_t node = p2g_tile_lds(lx + kx, ly + ky, lz);
                float4 t = slab[node];
                t.x += acc[q][0];
                t.y += acc[q][1];
                t.z += acc[q][2];
                t.w += acc[q][3];
                slab[node] = t;
                // The next step's nodes overlap other lanes' nodes of this one: its reads
                // come after these writes (a wave's LDS operations are carried out in
                // their order).
                __asm__ volatile("" ::: "memory");
            }
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < TILE_NODES; j += T) {
            const uint32_t x = j % 6u, y = (j / 6u) % 6u, z = j / 36u;
            float4 t = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (uint32_t w = 0; w < 3; w++) {
                if (z < w || z > w + 3u) continue;
#pragma unroll
                for (uint32_t p = 0; p < SUB; p++) {
                    const float4 u = S.slab[w + 3u * p][p2g_tile_lds(x, y, z - w)];
                    t.x += u.x;
                    t.y += u.y;
                    t.z += u.z;
                    t.w += u.w;
                }
            }
            E.tiles[(size_t)hid * TILE_NODES + tile_index(x, y, z)] = t;
        }
        if (wave == 0u) E.cell_cnt[(size_t)hid * NODES_PER_BLOCK + lane] = tot;
        if (threadIdx.x == 0u) E.in.rel[hid] = make_uint2((uint32_t)(rel >> 32), (uint32_t)rel);
        if constexpr (FAST)
            if (wave == 0u) finish_block(E.P, E.in, E.keys, hid, block_key, lane, range, br.total, seen);
    }
}

// The closest leaves of a block's nodes (lane = node, at cell_pos; those in `need`)
// for every trimesh collider into S.key, by the whole workgroup.
__device__ inline void mesh_queries(const Colliders &cs, const float4 *box, MeshShared &S, float h, float3 cell_pos,
                                    bool need) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float cap = h * 1.5f;
    for (uint32_t i = 0; i < cs.count; i++) {
        const float4 a = cs.shapes[2 * i];
        if (__float_as_uint(a.w) != 6u) continue;
        const float4 lo = box[2 * i], hi = box[2 * i + 1];
        const bool on = need && cell_pos.x >= lo.x && cell_pos.x <= hi.x && cell_pos.y >= lo.y && cell_pos.y <= hi.y &&
                        cell_pos.z >= lo.z && cell_pos.z <= hi.z;
        if (wave == 0u) {
            S.key[i][lane] = ~0ull;
            S.tie[lane] = ~0u;
        }
        if (__ballot(on) == 0ull) continue;  // (every wave holds the same nodes)
        const float4 rot = cs.poses[2 * i], ts = cs.poses[2 * i + 1];
        const uint32_t base = cs.mesh_base[i], count = __float_as_uint(a.z);
        const uint32_t search = cs.mesh_search[i];
        const bool flat = search == MESH_FLAT;
        const float4 *node = cs.mesh_nodes + 2u * (size_t)base, *leaf = cs.mesh_leaves + 3u * (size_t)base;
        const float3 pt = sim_inv_mul_pt(rot, ts, cell_pos);
        if (flat) {
            if (threadIdx.x == 0u) S.n_cand = 0u;
            __syncthreads();
        }
        if (search == MESH_WALK) {
            if (threadIdx.x == 0u) S.n_cand = SLOSH_NONE;
        } else if (flat || wave == 0u) {
            // The block's box in the mesh's frame, from its first node.
            const float3 w0 = make_float3(__shfl(cell_pos.x, 0), __shfl(cell_pos.y, 0), __shfl(cell_pos.z, 0));
            const float3 c = sim_inv_mul_pt(rot, ts, make_float3(w0.x + cap, w0.y + cap, w0.z + cap));
            const float4 inv = make_float4(-rot.x, -rot.y, -rot.z, rot.w);
            const float3 ix = quat_rotate(inv, make_float3(1.0f, 0.0f, 0.0f));
            const float3 iy = quat_rotate(inv, make_float3(0.0f, 1.0f, 0.0f));
            const float3 iz = quat_rotate(inv, make_float3(0.0f, 0.0f, 1.0f));
            const float s = 1.001f * cap / fabsf(ts.w);
            const float3 e = make_float3((fabsf(ix.x) + fabsf(iy.x) + fabsf(iz.x)) * s,
                                         (fabsf(ix.y) + fabsf(iy.y) + fabsf(iz.y)) * s,
                                         (fabsf(ix.z) + fabsf(iy.z) + fabsf(iz.z)) * s);
            const float size = fmaxf(fmaxf(fabsf(c.x), fabsf(c.y)), fabsf(c.z));
            const float reach = 1.001f * cap + 1.0e-5f * size;
            if (flat) mesh_candidates_flat(S, node, count, c, e, reach);
            else mesh_candidates(S, node, c, e, reach);
        }
        __syncthreads();
        // Nodes that are walked: 4 x 2 of them per wave (side by side, so that they visit much
        // the same).
        const bool mine = lane >> 3 == wave;
        const uint32_t n = S.n_cand;
        if (n > MESH_CAND) {
            if (on && mine) {
                const uint32_t lf = trimesh_walk(node, leaf, count, pt, cap, search != MESH_WALK);
                if (lf != SLOSH_NONE) S.key[i][lane] = mesh_key(0.0f, lf);
            }
        } else {
            // Every wave culls by the closest any of them has found so far. `eps`: above the
            // rounding of distances between numbers of the mesh's size.
            const float size = cs.mesh_size[i] + cap, eps = 3.0e-7f * size;
            volatile unsigned long long *closest = &S.key[i][lane];
            for (uint32_t q = wave; q < n; q += MESH_WAVES) {
                const uint32_t lf = __builtin_amdgcn_readfirstlane(S.cand[q]);
                const unsigned long long key = *closest;
                const float best = key == ~0ull ? cap : key_distance(key) + eps;
                if (on && box_distance(node[2u * lf], node[2u * lf + 1u], pt) <= best) {
                    float3 p;
                    uint32_t tri, feat, id;
                    const float4 *lv = leaf + 3u * (size_t)lf;
                    const float dist = leaf_distance(lv, pt, &p, &tri, &feat, &id);
                    if (dist <= fminf(best, cap)) {
                        const unsigned long long k = mesh_key(dist, lf);
                        // What was the closest before: of waves that come at once, each sees
                        // the one before it. (Its point may not be stored yet: then a node
                        // counts as tied without need, and is walked to the same result.)
                        const unsigned long long old = k < key ? atomicMin(&S.key[i][lane], k) : key;
                        volatile float *px = &S.point[0][lane], *py = &S.point[1][lane], *pz = &S.point[2][lane];
                        const float d = key_distance(old);  // (a NaN if there was none)
                        if (fabsf(d - dist) <= eps &&
                            fmaxf(fmaxf(fabsf(*px - p.x), fabsf(*py - p.y)), fabsf(*pz - p.z)) > eps) {
                            if (fmaxf(leaf_box_distance(lv, pt),
                                      leaf_box_distance(leaf + 3u * (size_t)key_leaf(old), pt)) >= dist - 2.0f * eps)
                                atomicMin(&S.tie[lane], __float_as_uint(fminf(d, dist)));
                        }
                        if (k < old) {
                            *px = p.x;
                            *py = p.y;
                            *pz = p.z;
                        }
                    }
                }
            }
            __syncthreads();
            if (on && mine) {
                const unsigned long long key = *closest;
                const float d = key_distance(key);
                bool decide = __uint_as_float(S.tie[lane]) <= d + eps;
                if (d + eps >= cap)
                    decide = decide || leaf_box_distance(leaf + 3u * (size_t)key_leaf(key), pt) >= d - eps;
                if (decide) {
                    const uint32_t lf = trimesh_walk(node, leaf, count, pt, fminf(cap, d + 4.0f * eps), true);
                    S.key[i][lane] = lf != SLOSH_NONE ? mesh_key(0.0f, lf) : ~0ull;
                }
            }
        }
        __syncthreads();
    }
}

// What the grid update prepares for the fused G2P kernel: each block's storage start
// and its items (ITEM_*, one per 64 consecutive entries of its sequence), from the
// regions' sums and the block's place in them, and cleared counters (output slots taken,
// stayers).
struct ItemLists {
    uint32_t *items;
    const unsigned long long *rsum;
    const uint2 *rel;
    uint32_t *blk_start, *taken, *stay, *n_items;
    uint32_t rshift;
};

// The next substep's table, reset here (`prime`).
struct NextTable {
    uint32_t *keys, *counters, *mlist, *ovf_slot, *ovf_hid;
    uint4 *arrive;  // per block: movers; slot, start and count of its stayers' range (else SLOSH_NONE)
    uint2 *rlist;
    uint32_t *rcnt;
    unsigned long long *rsum;
    uint32_t rshift, prime;
};

__device__ inline void reset_next_table(const NextTable &nt, uint32_t cap) {
    if (!nt.prime) return;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t s = i; s < cap; s += gridDim.x * blockDim.x) {
        nt.keys[s] = SLOSH_NONE;
        nt.arrive[s] = make_uint4(0u, SLOSH_NONE, 0u, 0u);
    }
    if (blockIdx.x == 0u && threadIdx.x < REGIONS) {
        nt.rcnt[threadIdx.x * RCNT_STRIDE] = 0u;
        nt.rsum[threadIdx.x * RSUM_STRIDE] = 0ull;
    }
    if (i == 0u) {
        nt.counters[CTR_NUM_BLOCKS] = 0u;
        nt.counters[CTR_OVERFLOW] = 0u;
    }
}

// mode 0: node momentum from tiles; mode 1: nodes already hold momentum (P2G hook).
// do_update 0: only combine tiles (grid update disabled; nothing to do to the nodes in mode 1).
template <bool MESH>
__global__ __launch_bounds__(MESH ? 64 * MESH_WAVES : 64) void k_grid_update(StepParams P, const float4 *__restrict__ tiles,
                                                     float4 *__restrict__ nodes, const uint32_t *__restrict__ nbr,
                                                     const uint32_t *__restrict__ keys, Colliders cs,
                                                     const NodeColl *__restrict__ coll_prev, NodeColl *__restrict__ coll_cur,
                                                     Members M, ItemLists L, NextTable nt, uint32_t mode,
                                                     uint32_t do_update) {
    const uint32_t *__restrict__ blk_cnt = M.blk_cnt;
    __shared__ float4 cbox[2 * SLOSH_MAX_COLLIDERS];
    if (threadIdx.x < cs.count) collider_box<MESH>(cs, threadIdx.x, 1.5f * P.h, &cbox[2 * threadIdx.x], &cbox[2 * threadIdx.x + 1]);
    __syncthreads();
    const uint32_t B = M.counters[CTR_NUM_BLOCKS];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const int x = lane & 3, y = (lane >> 2) & 3, z = lane >> 4;
    // Storage and items before the lane's region.
    const unsigned long long rs = L.rsum[lane * RSUM_STRIDE];
    const uint32_t up_p = wave_inclusive_scan((uint32_t)(rs >> 32)), up_i = wave_inclusive_scan((uint32_t)rs);
    if (mode == 0 && blockIdx.x == 0u && threadIdx.x == 0u) *L.n_items = __builtin_amdgcn_readlane(up_i, 63);
    // With trimesh colliders a workgroup shares one block: every wave holds its nodes
    // (and takes part in mesh_queries), the first one writes them.
    __shared__ typename std::conditional<MESH, MeshShared, char>::type shared;
    const uint32_t xcd = blockIdx.x & 7u, wg = blockIdx.x >> 3, wgs = gridDim.x >> 3;
    const bool owner = !MESH || wave == 0u;
    for (uint32_t j = wg;; j += wgs) {
        const uint32_t k = xcd_item(xcd, j, B);
        if (k >= B) break;
        const uint32_t hid = __builtin_amdgcn_readfirstlane(M.blist[k]);
        const uint32_t block_key = __builtin_amdgcn_readfirstlane(keys[hid]);
        // The neighbour table (lane l: entry l, see NBR_STRIDE).
        const uint32_t nb = lane < NBR_STRIDE ? nbr[(size_t)hid * NBR_STRIDE + lane] : SLOSH_NONE;
        const uint32_t prev = __builtin_amdgcn_readlane(nb, NBR_PREV);
        if (owner) {
            const BlockRange br = M.fast ? block_range<true>(M, hid) : block_range<false>(M, hid);
            const uint32_t n = item_count(br), r = hid >> L.rshift;
            // (Where its particles begin; a block without any, where its region's do.)
            uint32_t start = r ? __builtin_amdgcn_readlane(up_p, r - 1u) : 0u;
            if (n) {
                uint32_t item0;
                if (mode == 0) {
                    const uint2 rel = L.rel[hid];
                    item0 = rel.y + (r ? __builtin_amdgcn_readlane(up_i, r - 1u) : 0u);
                    start = M.fast ? start + rel.x : M.blk_start[hid];
                } else {
                    // A hook did P2G after a full sort: the items in order of arrival (their
                    // count was cleared by the sort).
                    uint32_t at = 0u;
                    if (lane == 0u) at = atomicAdd(L.n_items, n);
                    item0 = __builtin_amdgcn_readfirstlane(at);
                    start = M.blk_start[hid];
                }
                // Four items at a time, a word per lane.
                const uint32_t w = lane & 15u;
                uint32_t v = (uint32_t)__shfl((int)nb, (int)w);
                v = w == ITEM_HID ? hid : v;
                v = w == ITEM_CAND_LO ? br.cand_lo : v;
                v = w == ITEM_CAND_N ? br.cand_n : v;
                v = w == ITEM_LIST_N ? br.list_n : v;
                v = w == ITEM_START ? start : v;
                v = w == ITEM_KEY ? block_key : v;
                v = w == ITEM_TOTAL ? br.total : v;
                v = w == ITEM_OVERFLOW ? (br.overflow ? 1u : 0u) : v;
                for (uint32_t c = lane >> 4; c < n; c += 4u)
                    L.items[(size_t)(item0 + c) * ITEM_WORDS + w] = w == ITEM_FIRST ? 64u * c : v;
            }
            if (lane == 0u) {
                if (M.fast) L.blk_start[hid] = start;
                L.taken[hid] = 0u;
                L.stay[hid] = 0u;
            }
        }
        float4 acc;
        if (mode == 0) {
            // Tiles of blocks without particles were not written (they count as
            // zero). Each tile value is loaded together with its block's particle
            // count and then selected by it, so the tile loads wait only for the
            // neighbour ids, not for the counts (every tile lies inside the
            // allocation, written or not). The part of a "-1" neighbour's tile
            // that lands on this block is one contiguous region of that tile.
            float4 t[8];
            uint32_t c[8];
            t[0] = tiles[(size_t)hid * TILE_NODES + x + 4 * y + 16 * z];
            c[0] = blk_cnt[hid];
#pragma unroll
            for (int d = 1; d < 8; d++) {
                const int ox = ASSOC[d][0], oy = ASSOC[d][1], oz = ASSOC[d][2];
                t[d] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                c[d] = 0u;
                const uint32_t src = __builtin_amdgcn_readlane(nb, NBR_MINUS + d - 1);
                if ((ox == 0 || x <= 1) && (oy == 0 || y <= 1) && (oz == 0 || z <= 1)) {
                    if (src != SLOSH_NONE) {
                        t[d] = tiles[(size_t)src * TILE_NODES + tile_index(x + 4 * ox, y + 4 * oy, z + 4 * oz)];
                        c[d] = blk_cnt[src];
                    }
                }
            }
            acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (int d = 0; d < 8; d++) {
                // Bitwise select: a stale tile (possibly NaN) never enters the sum.
                const bool on = c[d] != 0u;
                const float4 v = make_float4(__uint_as_float(on ? __float_as_uint(t[d].x) : 0u),
                                             __uint_as_float(on ? __float_as_uint(t[d].y) : 0u),
                                             __uint_as_float(on ? __float_as_uint(t[d].z) : 0u),
                                             __uint_as_float(on ? __float_as_uint(t[d].w) : 0u));
                if (d == 0) {
                    acc = v;
                } else {
                    acc.x += v.x;
                    acc.y += v.y;
                    acc.z += v.z;
                    acc.w += v.w;
                }
            }
        } else {
            if (!do_update) continue;
            acc = nodes[(size_t)hid * NODES_PER_BLOCK + lane];
        }
        if (MESH) __syncthreads();  // every wave has read the nodes (mode 1) and is done with the last block
        if (!do_update) {
            if (owner) nodes[(size_t)hid * NODES_PER_BLOCK + lane] = acc;
            continue;
        }
        const float h = P.h, dt = P.dt;
        int bx, by, bz;
        uint32_t scene;
        unpack_key(P.batched, block_key, &bx, &by, &bz, &scene);
        float3 cell_pos = make_float3((float)(bx * 4 + x) * h, (float)(by * 4 + y) * h, (float)(bz * 4 + z) * h);
        // update_single_cell, grid_update.slang:154-163
        const float mass = acc.w;
        const float inv_mass = mass > 0.0f ? 1.0f / mass : 0.0f;
        const float lim = P.h_dt;
        float3 v;
        v.x = fminf(fmaxf((acc.x + mass * P.gravity[0] * dt) * inv_mass, -lim), lim);
        v.y = fminf(fmaxf((acc.y + mass * P.gravity[1] * dt) * inv_mass, -lim), lim);
        v.z = fminf(fmaxf((acc.z + mass * P.gravity[2] * dt) * inv_mass, -lim), lim);
        const unsigned long long(*mesh_keys)[NODES_PER_BLOCK] = nullptr;
        if constexpr (MESH) {
            mesh_queries(cs, cbox, shared, h, cell_pos,
                         P.coll_cache ? prev == SLOSH_NONE || coll_prev == nullptr : mass > 0.0f);
            if (!owner) continue;
            mesh_keys = shared.key;
        }
        if (cs.count > 0) {
            NodeColl c;
            bool have = true;
            if (P.coll_cache) {
                if (prev != SLOSH_NONE && coll_prev != nullptr) c = coll_prev[(size_t)prev * NODES_PER_BLOCK + lane];
                else c = collide<MESH>(cs, cbox, h, cell_pos, mesh_keys, lane);
                coll_cur[(size_t)hid * NODES_PER_BLOCK + lane] = c;
            } else if (mass > 0.0f) {
                // Static colliders: the cached record equals a fresh collide(); a
                // zero-mass node has v = 0, which every boundary condition keeps.
                c = collide<MESH>(cs, cbox, h, cell_pos, mesh_keys, lane);
            } else {
                have = false;
            }
            if (have && __float_as_uint(c.point_valid.w) != 0u) {
                uint2 bc = cs.mats[__float_as_uint(c.normal_id.w)];
                float3 n = make_float3(c.normal_id.x, c.normal_id.y, c.normal_id.z);
                float3 dd = make_float3(cell_pos.x - c.point_valid.x, cell_pos.y - c.point_valid.y,
                                        cell_pos.z - c.point_valid.z);
                float dist = (dd.x * n.x + dd.y * n.y + dd.z * n.z) - h;
                v = project_velocity(bc, v, n, dist, dt);
            }
        }
        nodes[(size_t)hid * NODES_PER_BLOCK + lane] = make_float4(v.x, v.y, v.z, mass);
    }
    reset_next_table(nt, P.cap);
}

// A BVH in the layout of the grid update: per node its box with the entry link (all ones: a
// leaf) and the exit link in the spare components, and for a leaf its triangle's vertices
// with the triangle's index. A leaf's box is that of its triangle (the walk never reads a
// leaf's own), grown by 1 % of its extent and well above the rounding of its coordinates.
// (Packed on the host and uploaded, a mesh of 44402 triangles took 1.6 ms to set, now 1.1.)
__global__ __launch_bounds__(256) void k_pack_mesh(const float4 *__restrict__ vtx, const uint32_t *__restrict__ idx,
                                                   uint32_t count, float4 *__restrict__ nodes,
                                                   float4 *__restrict__ leaves) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    const uint32_t entry = idx[3u * (size_t)k], exit_ = idx[3u * (size_t)k + 1u], tri = idx[3u * (size_t)k + 2u];
    float4 lo = vtx[2u * (size_t)k], hi = vtx[2u * (size_t)k + 1u];
    if (entry == SLOSH_NONE) {
        const uint32_t *t = idx + 3u * (size_t)count + 3u * (size_t)tri;
        const float4 *v = vtx + 2u * (size_t)count;
        const float4 a = v[t[0]], b = v[t[1]], c = v[t[2]];
        const float w = __uint_as_float(tri);
        float4 *leaf = leaves + 3u * (size_t)k;
        leaf[0] = make_float4(a.x, a.y, a.z, w);
        leaf[1] = make_float4(b.x, b.y, b.z, w);
        leaf[2] = make_float4(c.x, c.y, c.z, w);
        lo = make_float4(fminf(fminf(a.x, b.x), c.x), fminf(fminf(a.y, b.y), c.y), fminf(fminf(a.z, b.z), c.z), 0.0f);
        hi = make_float4(fmaxf(fmaxf(a.x, b.x), c.x), fmaxf(fmaxf(a.y, b.y), c.y), fmaxf(fmaxf(a.z, b.z), c.z), 0.0f);
        const float extent = fmaxf(fmaxf(hi.x - lo.x, hi.y - lo.y), hi.z - lo.z);
        const float size = fmaxf(fmaxf(fmaxf(fabsf(lo.x), fabsf(hi.x)), fmaxf(fabsf(lo.y), fabsf(hi.y))),
                                 fmaxf(fabsf(lo.z), fabsf(hi.z)));
        const float grow = 0.01f * extent + 1.0e-5f * size;
        lo = make_float4(lo.x - grow, lo.y - grow, lo.z - grow, 0.0f);
        hi = make_float4(hi.x + grow, hi.y + grow, hi.z + grow, 0.0f);
    }
    nodes[2u * (size_t)k] = make_float4(lo.x, lo.y, lo.z, __uint_as_float(entry));
    nodes[2u * (size_t)k + 1u] = make_float4(hi.x, hi.y, hi.z, __uint_as_float(exit_));
}

struct Bodies {
    float4 *poses;        // 2 per body
    float4 *vels;         // 2 per body: linear, angular
    const float4 *mprops; // 5 per body: inv_inertia rows 0..2, inv_mass, com (world)
    const float4 *local_com; // 1 per body
    int *impulses;        // 6 per body: linear xyz, angular xyz (fixed point x 1e5)
    uint32_t count;
};

__device__ inline float len3(float3 a) { return sqrtf(a.x * a.x + a.y * a.y + a.z * a.z); }

// rigid_impulses.slang:70-121 with body.slang:63-130, for body `id`.
__device__ void integrate_body(const StepParams &P, const Bodies &b, uint32_t id) {
    const float dt = P.dt;
    float3 lin, ang;
    lin.x = (float)b.impulses[6 * id + 0] / 1.0e5f;
    lin.y = (float)b.impulses[6 * id + 1] / 1.0e5f;
    lin.z = (float)b.impulses[6 * id + 2] / 1.0e5f;
    ang.x = (float)b.impulses[6 * id + 3] / 1.0e5f;
    ang.y = (float)b.impulses[6 * id + 4] / 1.0e5f;
    ang.z = (float)b.impulses[6 * id + 5] / 1.0e5f;
#pragma unroll
    for (int k = 0; k < 6; k++) b.impulses[6 * id + k] = 0;
    const float4 ii0 = b.mprops[5 * id + 0], ii1 = b.mprops[5 * id + 1], ii2 = b.mprops[5 * id + 2];
    const float4 im = b.mprops[5 * id + 3];
    float4 vl = b.vels[2 * id], va = b.vels[2 * id + 1];
    float3 nl = make_float3(vl.x + im.x * lin.x, vl.y + im.y * lin.y, vl.z + im.z * lin.z);
    float3 na = make_float3(va.x + (ang.x * ii0.x + ang.y * ii1.x + ang.z * ii2.x),
                            va.y + (ang.x * ii0.y + ang.y * ii1.y + ang.z * ii2.y),
                            va.z + (ang.x * ii0.z + ang.y * ii1.z + ang.z * ii2.z));
    float ln = len3(nl), an = len3(na);
    float lin_limit = 0.1f * P.h / dt;
    if (len3(lin) != 0.0f || len3(ang) != 0.0f) {
        if (ln > lin_limit) nl = make_float3(nl.x * (lin_limit / ln), nl.y * (lin_limit / ln), nl.z * (lin_limit / ln));
        if (an > 1.0f) na = make_float3(na.x * (1.0f / an), na.y * (1.0f / an), na.z * (1.0f / an));
    }
    // integrate_velocity
    float4 rot = b.poses[2 * id], ts = b.poses[2 * id + 1];
    float4 lc = b.local_com[id];
    float3 init_com = sim_mul_pt(rot, ts, make_float3(lc.x, lc.y, lc.z));
    float3 sa = make_float3(na.x * dt, na.y * dt, na.z * dt);
    float angle = len3(sa);
    float4 dq = make_float4(0.0f, 0.0f, 0.0f, 1.0f);
    if (angle != 0.0f) {
        float s = sinf(angle * 0.5f) / angle;
        dq = make_float4(sa.x * s, sa.y * s, sa.z * s, cosf(angle * 0.5f));
    }
    float3 rr = quat_rotate(dq, make_float3(ts.x - init_com.x, ts.y - init_com.y, ts.z - init_com.z));
    float4 nq;
    nq.x = dq.w * rot.x + dq.x * rot.w + dq.y * rot.z - dq.z * rot.y;
    nq.y = dq.w * rot.y - dq.x * rot.z + dq.y * rot.w + dq.z * rot.x;
    nq.z = dq.w * rot.z + dq.x * rot.y - dq.y * rot.x + dq.z * rot.w;
    nq.w = dq.w * rot.w - dq.x * rot.x - dq.y * rot.y - dq.z * rot.z;
    float sq = nq.x * nq.x + nq.y * nq.y + nq.z * nq.z + nq.w * nq.w;
    float k = 0.5f * (3.0f - sq);
    b.poses[2 * id] = make_float4(nq.x * k, nq.y * k, nq.z * k, nq.w * k);
    b.poses[2 * id + 1] = make_float4(init_com.x + rr.x * ts.w + nl.x * dt, init_com.y + rr.y * ts.w + nl.y * dt,
                                      init_com.z + rr.z * ts.w + nl.z * dt, ts.w);
    nl.x += P.gravity[0] * (im.x != 0.0f ? 1.0f : 0.0f) * dt;
    nl.y += P.gravity[1] * (im.y != 0.0f ? 1.0f : 0.0f) * dt;
    nl.z += P.gravity[2] * (im.z != 0.0f ? 1.0f : 0.0f) * dt;
    b.vels[2 * id] = make_float4(nl.x, nl.y, nl.z, 0.0f);
    b.vels[2 * id + 1] = make_float4(na.x, na.y, na.z, 0.0f);
}


__global__ void k_rigid_update(StepParams P, Bodies b) {
    if (threadIdx.x < b.count) integrate_body(P, b, threadIdx.x);
}

__device__ inline void load_halo(float4 *__restrict__ sh, const float4 *__restrict__ nodes,
                                 const uint32_t *__restrict__ nbr, uint32_t hid) {
    for (uint32_t j = threadIdx.x; j < TILE_NODES; j += blockDim.x) {
        uint32_t sx = j % 6u, sy = (j / 6u) % 6u, sz = j / 36u;
        uint32_t ox = sx >= 4u, oy = sy >= 4u, oz = sz >= 4u;
        uint32_t oi = ox * 4u + oy * 2u + oz;
        uint32_t src = oi == 0u ? hid : nbr[(size_t)hid * NBR_STRIDE + oi - 1u];
        uint32_t node = (sx - 4u * ox) + 4u * (sy - 4u * oy) + 16u * (sz - 4u * oz);
        sh[j] = src != SLOSH_NONE ? nodes[(size_t)src * NODES_PER_BLOCK + node] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

// The same by one wave into its own LDS tile: lanes 0..6 hold the neighbour ids, lane 7
// the block's, and each lane takes its nodes' from them.
__device__ inline void load_halo_wave(float4 *__restrict__ sh, const float4 *__restrict__ nodes, uint32_t nb,
                                      uint32_t lane) {
    constexpr uint32_t R = (TILE_NODES + 63u) / 64u;
    float4 v[R];
#pragma unroll
    for (uint32_t r = 0; r < R; r++) {
        const uint32_t j = lane + 64u * r;
        const uint32_t sx = j % 6u, sy = (j / 6u) % 6u, sz = j / 36u;
        const uint32_t ox = sx >= 4u, oy = sy >= 4u, oz = sz >= 4u;
        const uint32_t oi = ox * 4u + oy * 2u + oz;
        const uint32_t src = (uint32_t)__shfl((int)nb, oi == 0u ? 7 : (int)oi - 1);
        const uint32_t node = (sx - 4u * ox) + 4u * (sy - 4u * oy) + 16u * (sz - 4u * oz);
        v[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (j < TILE_NODES && src != SLOSH_NONE) v[r] = nodes[(size_t)src * NODES_PER_BLOCK + node];
    }
#pragma unroll
    for (uint32_t r = 0; r < R; r++) {
        const uint32_t j = lane + 64u * r;
        if (j < TILE_NODES) sh[j] = v[r];
    }
}

// What the fused G2P kernel counts per block of this table: output slots handed out
// and particles that stay. For the next substep it inserts the blocks into NextTable
// and appends the particles that leave their block to their new block's list.
struct NextSort {
    uint32_t *taken, *stay;
    uint32_t *errors;         // this substep's error word (ERR_KEY_RANGE)
};

// F64: the SVD-based steps refined to FP64 accuracy. The bounds keep that variant of
// every material at three waves per SIMD (168 VGPRs), the others at four or more.
//
// One wave per item, in a workgroup of its own: 64 consecutive entries of a block's
// sequence, with the block's node halo in an LDS tile, so that waves share no barrier
// and a block's last, partly filled round holds one wave instead of a workgroup. With
// one workgroup per block a second round of 256 entries cost a block 3.8 us of serial
// latency, and a block of 50 particles kept four waves; per wave (medians of the kernel,
// before and after): 2.1M sand and spheres (42k blocks) 643 -> 252 us, 48 scenes of
// three materials (2.0M) 320 -> 156 us, sand on a heightfield (85k) 43 -> 19 us, dam
// break of 131k 15.7 -> 13.1 us and of 1M 66 -> 46 us once it moves. (Four items to a
// workgroup kept the registers of its finished waves idle until the last one ended and
// put a small scene's waves on a quarter of the CUs: 266, 168 and, 8k particles of four
// materials, 29 us against 19.) The small scenes are bound by the chain of dependent
// loads and the ~1000 instructions of one particle, 1M by memory (188 MB per launch),
// FP64 materials by latency at three waves per SIMD and half by issue.
//
// Output order: a block's members take the output slots [start, start + total)
// of the block in order of arrival of their waves (one atomic per wave, issued
// before the sums that hide it), so a block's particles stay together in
// storage. The particles whose updated position leaves the block join their new
// block's list in the next substep's table; the others are counted (the block's
// stayers).
// The arguments, read where they are used: held in scalar registers from the start
// 118 of them spilled to VGPR lanes. late_args() gives the compiler a new, opaque address
// of the kernel's argument block, so that what is read through it is loaded after that
// point: the neo-Hookean instance went from 108 to 93 VGPRs (now 77: six waves per SIMD
// instead of four; 1M particles 53.0 -> 48.6 us), the FP32 one of every material from 145
// to 128 (now 99).
struct G2pArgs {
    StepParams P;
    PBuf in, out;
    PStatic st;
    uint32_t pcap;
    float *fdt;
    NextTable nt;
    NextSort ns;
    Bodies bodies;
};

template <uint32_t MODELS, bool F64>
__global__ __launch_bounds__(64, F64 && MODELS != 3u ? 3 : 4) void k_g2p_update(G2pArgs args, Members M,
                                                    const uint32_t *__restrict__ items,
                                                    const float4 *__restrict__ nodes) {
    __shared__ float4 sh[TILE_NODES];
    // The FP64 corotated instance fits four waves per SIMD (128 VGPRs) without scratch
    // memory, whose set-up alone costs more than the fourth wave gains, if it recomputes and
    // stashes more (1.2M corotated particles 119.3 -> 114.3 us a substep; the neo-Hookean
    // instance lost 2 us of 92 at 1M by the same).
    constexpr bool TIGHT = F64 && MODELS == 3u;
    // integrate_bodies: reads no particle or grid state (the impulses it applies
    // are only written by the host), so the last workgroup runs it alongside the
    // particle update.
    if (blockIdx.x == gridDim.x - 1u) {  // (the one beyond the eight ranges' workgroups)
        if (threadIdx.x < args.bodies.count) integrate_body(args.P, args.bodies, threadIdx.x);
        return;
    }
    const uint32_t n_items = M.counters[CTR_ITEMS];
    for (uint32_t j = blockIdx.x >> 3;; j += gridDim.x >> 3) {
        const uint32_t i = xcd_item(blockIdx.x & 7u, j, n_items);
        if (i >= n_items) break;
        // Opaque copies of the lane, for the item and for each round over its entries:
        // nearly every wave goes round once, so little is worth computing ahead of the
        // loops and holding in registers (the halo's addresses alone took 15).
        uint32_t lane1 = threadIdx.x;
        asm volatile("" : "+v"(lane1));
        const uint32_t item = items[(size_t)i * ITEM_WORDS + (lane1 & 15u)];
        const uint32_t hid = __builtin_amdgcn_readlane(item, ITEM_HID);
        const uint32_t first = __builtin_amdgcn_readlane(item, ITEM_FIRST);
        const uint32_t s0 = __builtin_amdgcn_readlane(item, ITEM_START);
        const uint32_t block_key = __builtin_amdgcn_readlane(item, ITEM_KEY);
        const uint32_t total = __builtin_amdgcn_readlane(item, ITEM_TOTAL);
        BlockRange br;
        br.cand_lo = __builtin_amdgcn_readlane(item, ITEM_CAND_LO);
        br.cand_n = __builtin_amdgcn_readlane(item, ITEM_CAND_N);
        br.list = M.fast ? M.mlist + (size_t)hid * MOVER_CAP : M.perm + s0;
        br.list_n = __builtin_amdgcn_readlane(item, ITEM_LIST_N);
        // The item's entries (a candidate is a member only if it is still in the
        // block); the block's first item then takes the overflow list, only if some
        // of the block's movers overflowed theirs (entries of other blocks are
        // skipped). Per member: G2P, update, output at the next free slot of the
        // block's range, listed if it leaves the block, its blocks inserted into the
        // next table. Every lane runs the same number of iterations (the wave-level
        // counting and run detection see all lanes).
        const uint32_t n_main = br.cand_n + br.list_n;
        const uint32_t n_ovf =
            first == 0u && __builtin_amdgcn_readlane(item, ITEM_OVERFLOW) ? M.counters[CTR_OVERFLOW] : 0u;
        for (uint32_t o = 0; o < 64u + n_ovf; o += 64u) {
            const G2pArgs &A = late_args<G2pArgs>();
            uint32_t lane2 = TIGHT ? threadIdx.x : lane1;
            asm volatile("" : "+v"(lane2));
            const uint32_t lane = TIGHT ? lane2 : lane1;
            bool entry;
            uint32_t p = 0u;
            if (o == 0u) {
                const uint32_t m = first + lane;
                entry = m < n_main;
                if (entry) p = entry_slot(br, m);
            } else {
                const uint32_t q = o - 64u + lane;
                entry = q < n_ovf && M.ovf_hid[q] == hid;
                if (entry) p = M.ovf_slot[q];
            }
            float4 ps = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            // The neo-Hookean-only instance has registers to spare: it issues the
            // deformation gradient and id loads with the position load (nearly
            // every entry is a member), the others after the G2P sums.
            constexpr bool EARLY = MODELS == 2u;
            float F[9];
            uint32_t oid = 0u;
            if (entry) {
                ps = A.in.pos[p];
                if (EARLY) {
#pragma unroll
                    for (int q = 0; q < 9; q++) F[q] = A.in.F[(size_t)q * A.pcap + p];
                    oid = A.in.ids[p];
                }
            }
            load_halo_wave(sh, nodes, item, lane2);  // (the last iteration may have reused the tile)
            const uint32_t wbits = __float_as_uint(ps.w);
            const uint32_t scene = wbits >> 1;
            const Stencil at = stencil_of(A.P.h, ps.x, ps.y, ps.z);
            int blk[3];
            uint32_t lc[3];
            block_of_cell(at.cell, blk, lc);
            const bool valid = entry && pack_key(A.P.batched, scene, blk[0], blk[1], blk[2]) == block_key;
            const uint64_t vmask = __ballot(valid);
            if (vmask == 0ull) continue;
            uint32_t ob = 0u;
            if (lane == 0) ob = atomicAdd(&A.ns.taken[hid], (uint32_t)__popcll(vmask));
            const float3 pos = make_float3(ps.x, ps.y, ps.z);
            float3 v;
            float aff[9], vgd;
            if (valid) g2p_particle(sh, A.P.h, A.P.inv_d, at, lc, (wbits & 1u) != 0u, &v, aff, &vgd);
            // The wave's first slot, from lane 0 (every lane is active here).
            const uint32_t out0 = __builtin_amdgcn_readfirstlane(ob);
            const uint32_t slot = s0 + out0 + (uint32_t)__popcll(vmask & lanemask_lt());
            uint32_t next_key = 0u;
            bool in_range = true;
            if (valid) {
                const G2pArgs &U = late_args<G2pArgs>();
                const StepParams &P = U.P;
                const PBuf &in = U.in, &out = U.out;
                const PStatic &st = U.st;
                const uint32_t pcap = U.pcap;
                float *const fdt = U.fdt;
                // Uniform masses (one for all, or one per scene) skip the 16-byte
                // velocity / mass load (the velocity comes from the grid): only the
                // update disables, and it zeroes the mass.
                const float mass = P.mass_uniform ? ((wbits & 1u) ? P.u_mass : 0.0f)
                                   : P.scene_mass  ? ((wbits & 1u) ? st.scene_rec[4 * (size_t)scene + 3].z : 0.0f)
                                                   : in.vm[p].w;
                if (!EARLY) {
#pragma unroll
                    for (int q = 0; q < 9; q++) F[q] = in.F[(size_t)q * pcap + p];
                    oid = in.ids[p];
                }
                float4 prop, model;
                static_records(P, st, oid, scene, &prop, &model);
                float3 np;
                advance_particle(P, pos, v, aff, F, prop, &np);
                // What is known before the stress leaves the registers: stored for a
                // particle that stays enabled (rewritten below if it does not).
                out.pos[slot] = make_float4(np.x, np.y, np.z, ps.w);
                out.vm[slot] = make_float4(v.x, v.y, v.z, mass);
                out.vgd[slot] = vgd;
                out.ids[slot] = oid;
                if (P.has_force) {
                    fdt[slot] = 0.0f;
                    fdt[(size_t)pcap + slot] = 0.0f;
                    fdt[2 * (size_t)pcap + slot] = 0.0f;
                }
                bool ok = np.x == np.x && np.y == np.y && np.z == np.z;
                int nx, ny, nz;
                uint32_t cell;
                assoc_block_cell(P.h, np.x, np.y, np.z, &nx, &ny, &nz, &cell);
                next_key = pack_key(P.batched, scene, nx, ny, nz);
                in_range = block_in_key_range(P.batched, nx, ny, nz);
                // The FP64 steps need the registers: the velocity gradient waits in
                // the wave's LDS tile, which the sums above no longer need.
                float *keep = reinterpret_cast<float *>(sh) + lane;
                float left_mass = mass, volume = prop.x;
                if (F64) {
#pragma unroll
                    for (int q = 0; q < 9; q++) keep[64 * q] = aff[q];
                }
                if (TIGHT) {
                    keep[64 * 9] = mass;
                    keep[64 * 10] = prop.x;
                    keep[64 * 11] = __uint_as_float(next_key);
                    keep[64 * 12] = __uint_as_float(p);
                }
                // Only Drucker-Prager particles read or write their plastic state
                // (the other particles' state slots are never read).
                const uint32_t tag = __float_as_uint(model.x);
                const bool plastic = P.has_sand && (tag == 2u || tag == 3u);
                float dps[3] = {0.0f, 0.0f, 0.0f}, stress[9];
                if (plastic) {
#pragma unroll
                    for (int q = 0; q < 3; q++) dps[q] = in.dps[(size_t)q * pcap + p];
                }
                material_update<MODELS, F64>(P, F, model, st, oid, scene, dps, stress);
                if (plastic) {
#pragma unroll
                    for (int q = 0; q < 3; q++) out.dps[(size_t)q * pcap + slot] = dps[q];
                }
                ok = ok && det3(F) > 0.0f;
                uint32_t from = p;
                if (F64) {
#pragma unroll
                    for (int q = 0; q < 9; q++) aff[q] = keep[64 * q];
                }
                if (TIGHT) {
                    left_mass = keep[64 * 9];
                    volume = keep[64 * 10];
                    next_key = __float_as_uint(keep[64 * 11]);
                    from = __float_as_uint(keep[64 * 12]);
                }
                finish_particle(P, ok, left_mass, volume, stress, aff, F);
#pragma unroll
                for (int q = 0; q < 9; q++) {
                    out.C[(size_t)q * pcap + slot] = aff[q];
                    out.F[(size_t)q * pcap + slot] = F[q];
                }
                if (!ok) {
                    const float4 old = in.pos[from];
                    out.pos[slot] = make_float4(old.x, old.y, old.z, __uint_as_float(wbits & ~1u));
                    out.vm[slot] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    next_key = block_key;
                }
            }
            const G2pArgs &N = late_args<G2pArgs>();
            const NextTable &nt = N.nt;
            const bool mover = valid && next_key != block_key;
            const uint64_t sm = __ballot(valid && !mover);
            uint32_t before = 1u;
            if (sm && lane == 0) before = atomicAdd(&N.ns.stay[hid], (uint32_t)__popcll(sm));
            const uint64_t mv = __ballot(mover);
            if (mv) {
                // Only a particle that leaves its block can leave the key space (a
                // block outside it would alias another one): reported, once per wave.
                const uint64_t bad = __ballot(mover && !in_range);
                if (bad && lane == 0) atomicOr(N.ns.errors, ERR_KEY_RANGE);
            }
            if (nt.prime) {
                // touch_primary_blocks and touch_neighbor_blocks of the next
                // substep (sort.slang:50-92). Particles that stay in this block
                // only flag it: its 8 blocks are inserted once, by the block's first
                // wave to arrive if it has stayers, else by the first wave that has (the
                // first one need not wait for the stayers' count). The others insert
                // theirs, one round per run of equal keys, and join their new block's
                // list, one atomic per run. Atomics on what every XCD writes take ~1 us
                // each: the chain is the insertion, then the list places, at once.
                BlockInit init{};
                init.list = nt.rlist;
                init.rcnt = nt.rcnt;
                init.rshift = nt.rshift;
                ListEntry entry;
                const uint64_t rheads = run_heads(next_key, mover);
                const bool opener = out0 == 0u && sm;
                const uint64_t self = opener ? sm & (0ull - sm) : 0ull;
                const uint64_t heads = (rheads & mv) | self;
                uint32_t own = SLOSH_NONE;
                if (heads) {
                    own = insert_blocks(nt.keys, N.P.cap, N.P.batched, next_key, heads, nt.counters, init, entry);
                    const int head = run_head_of(rheads);
                    const uint32_t to = __shfl(own, head);
                    const bool listed = mover && to != SLOSH_NONE;
                    uint32_t r0 = 0u;
                    if (listed && (int)lane == head) r0 = atomicAdd(&nt.arrive[to].x, run_length(rheads));
                    store_entry(init, entry);
                    const uint32_t r = __shfl(r0, head) + (lane - (uint32_t)head);
                    const bool over = listed && r >= MOVER_CAP;
                    if (listed && !over) nt.mlist[(size_t)to * MOVER_CAP + r] = slot;
                    const uint64_t om = __ballot(over);
                    if (om) {
                        uint32_t q0 = 0u;
                        if (lane == 0u) q0 = atomicAdd(&nt.counters[CTR_OVERFLOW], (uint32_t)__popcll(om));
                        q0 = __builtin_amdgcn_readfirstlane(q0);
                        if (over) {
                            const uint32_t q = q0 + (uint32_t)__popcll(om & lanemask_lt());
                            nt.ovf_slot[q] = slot;
                            nt.ovf_hid[q] = to;
                        }
                    }
                }
                bool mine = (self >> lane) & 1ull;
                if (!opener && __builtin_amdgcn_readfirstlane(before) == 0u) {
                    own = insert_blocks(nt.keys, N.P.cap, N.P.batched, block_key, 1ull, nt.counters, init, entry);
                    store_entry(init, entry);
                    mine = lane == 0u;
                }
                // Where the block's range is found again: by whoever inserted it, with
                // the same values.
                if (mine && own != SLOSH_NONE) {
                    uint32_t *a = &nt.arrive[own].x;
                    a[1] = hid;
                    a[2] = s0;
                    a[3] = total;
                }
            }
        }
    }
}

// WgTimestepBounds (timestep_bound.slang:18-92): per enabled particle, the
// material's P-wave sound-speed bound cfl h / max(|v|, c) (models/utils.slang:
// 119-135; elastic part of sand models, default.slang:94-127) and the velocity
// bound h / |v|, as the u32 fixed point of GpuTimestepBounds::secs_to_int,
// reduced with atomicMin into *out.
__device__ inline uint32_t secs_to_int(float secs) {
    const float x = floorf(secs * 1.0e12f);
    if (!(x > 0.0f)) return 0u;
    if (x >= 4294967295.0f) return 0xffffffffu;
    return (uint32_t)x;
}

// The bound of particle i (0xffffffff for a disabled particle).
__device__ inline uint32_t particle_dt_bound(const StepParams &P, const PBuf &buf, const PStatic &st, uint32_t pcap,
                                             uint32_t i) {
#pragma clang fp contract(off)
    const float h = P.h;
    const float4 ps = buf.pos[i];
    if ((__float_as_uint(ps.w) & 1u) == 0u) return 0xffffffffu;
    const float4 vm = buf.vm[i];
    const uint32_t oid = buf.ids[i];
    float4 prop, model;
    static_records(P, st, oid, __float_as_uint(ps.w) >> 1, &prop, &model);
    float F[9];
#pragma unroll
    for (int k = 0; k < 9; k++) F[k] = buf.F[(size_t)k * pcap + i];
    const float speed = sqrtf(vm.x * vm.x + vm.y * vm.y + vm.z * vm.z);
    float dt = 0.0f;
    if (__float_as_uint(model.x) < 4u) {
        const float lambda = model.y, mu = model.z, cfl = model.w;
        const float bulk = lambda + 2.0f * mu / 3.0f;
        const float shear = mu;
        const float density0 = vm.w / prop.x;
        const float curr_density = density0 / fmaxf(det3(F), 1.0e-6f);
        const float sound_speed = sqrtf((bulk + shear * 4.0f / 3.0f) / curr_density);
        dt = cfl * h / fmaxf(speed, sound_speed);
    }
    dt = fminf(dt, h / speed);
    return secs_to_int(dt);
}

__device__ inline uint32_t wave_min_u32(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, o));
    return v;
}

__global__ __launch_bounds__(256) void k_timestep_bound(StepParams P, PBuf buf, PStatic st, uint32_t pcap,
                                                        uint32_t *__restrict__ out) {
    uint32_t best = 0xffffffffu;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < P.n; i += gridDim.x * blockDim.x)
        best = min(best, particle_dt_bound(P, buf, st, pcap, i));
    best = wave_min_u32(best);
    if (lane_id() == 0 && best != 0xffffffffu) atomicMin(out, best);
}

// The same bound in two passes with no atomics and nothing to clear first:
// workgroup g stores the minimum over particles [g * TSB_CHUNK, (g + 1) *
// TSB_CHUNK) into partials[g] (0xffffffff if none is enabled), then one
// workgroup stores the minimum of the partials into *out. Integer minima, so
// the result is bit-identical to k_timestep_bound's.
__global__ __launch_bounds__(256) void k_timestep_bound_partials(StepParams P, PBuf buf, PStatic st, uint32_t pcap,
                                                                 uint32_t *__restrict__ partials) {
    __shared__ uint32_t wmin[4];
    uint32_t best = 0xffffffffu;
    const uint32_t base = blockIdx.x * TSB_CHUNK;
    const uint32_t end = min(P.n, base + TSB_CHUNK);
    for (uint32_t i = base + threadIdx.x; i < end; i += 256) best = min(best, particle_dt_bound(P, buf, st, pcap, i));
    best = wave_min_u32(best);
    if (lane_id() == 0) wmin[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) partials[blockIdx.x] = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
}

__global__ __launch_bounds__(256) void k_min_partials(const uint32_t *__restrict__ partials, uint32_t count,
                                                      uint32_t *__restrict__ out) {
    __shared__ uint32_t wmin[4];
    uint32_t best = 0xffffffffu;
    for (uint32_t i = threadIdx.x; i < count; i += 256) best = min(best, partials[i]);
    best = wave_min_u32(best);
    if (lane_id() == 0) wmin[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) *out = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
}

// G2P only, in place (hook path): writes velocity, velocity gradient, vel_grad_det.
__global__ __launch_bounds__(256) void k_g2p(StepParams P, PBuf buf, uint32_t pcap, const uint32_t *__restrict__ perm,
                                             const uint32_t *__restrict__ blist,
                                             const uint32_t *__restrict__ blk_start,
                                             const uint32_t *__restrict__ blk_cnt, const uint32_t *__restrict__ nbr,
                                             const float4 *__restrict__ nodes, const uint32_t *__restrict__ counters) {
    __shared__ float4 sh[TILE_NODES];
    const uint32_t B = counters[CTR_NUM_BLOCKS];
    for (uint32_t k = blockIdx.x; k < B; k += gridDim.x) {
        const uint32_t hid = blist[k];
        const uint32_t s0 = blk_start[hid], cnt = blk_cnt[hid];
        if (cnt == 0) continue;
        load_halo(sh, nodes, nbr, hid);
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < cnt; j += blockDim.x) {
            const uint32_t p = perm[s0 + j];
            const float4 ps = buf.pos[p];
            float3 v;
            float g[9];
            float vgd;
            const Stencil at = stencil_of(P.h, ps.x, ps.y, ps.z);
            int b[3];
            uint32_t lc[3];
            block_of_cell(at.cell, b, lc);
            g2p_particle(sh, P.h, P.inv_d, at, lc, (__float_as_uint(ps.w) & 1u) != 0u, &v, g, &vgd);
            float4 o = buf.vm[p];
            buf.vm[p] = make_float4(v.x, v.y, v.z, o.w);
#pragma unroll
            for (int k = 0; k < 9; k++) buf.C[(size_t)k * pcap + p] = g[k];
            buf.vgd[p] = vgd;
        }
        __syncthreads();
    }
}

// Particle update only, in place (hook path), over every particle.
template <uint32_t MODELS, bool F64>
__global__ __launch_bounds__(256, F64 ? 3 : 1) void k_particle_update(StepParams P, PBuf buf, PStatic st, uint32_t pcap,
                                                         float *__restrict__ fdt) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P.n) return;
    const float4 ps = buf.pos[p];
    const uint32_t wbits = __float_as_uint(ps.w);
    uint32_t enabled = wbits & 1u;
    float3 pos = make_float3(ps.x, ps.y, ps.z);
    float4 vmv = buf.vm[p];
    float3 v = make_float3(vmv.x, vmv.y, vmv.z);
    float mass = vmv.w;
    float aff[9], F[9];
#pragma unroll
    for (int k = 0; k < 9; k++) {
        aff[k] = buf.C[(size_t)k * pcap + p];
        F[k] = buf.F[(size_t)k * pcap + p];
    }
    const uint32_t oid = buf.ids[p];
    float dps[3] = {0.0f, 0.0f, 0.0f};
    if (P.has_sand) {
#pragma unroll
        for (int k = 0; k < 3; k++) dps[k] = buf.dps[(size_t)k * pcap + p];
    }
    float4 prop, model;
    static_records(P, st, oid, wbits >> 1, &prop, &model);
    float3 np;
    float stress[9];
    advance_particle(P, pos, v, aff, F, prop, &np);
    material_update<MODELS, F64>(P, F, model, st, oid, wbits >> 1, dps, stress);
    const bool ok = stays_enabled(np, F);
    finish_particle(P, ok, mass, prop.x, stress, aff, F);
    if (ok) {
        pos = np;
    } else {
        enabled = 0u;
        v = make_float3(0.0f, 0.0f, 0.0f);
        mass = 0.0f;
    }
    buf.pos[p] = make_float4(pos.x, pos.y, pos.z, __uint_as_float((wbits & ~1u) | enabled));
    buf.vm[p] = make_float4(v.x, v.y, v.z, mass);
#pragma unroll
    for (int k = 0; k < 9; k++) {
        buf.C[(size_t)k * pcap + p] = aff[k];
        buf.F[(size_t)k * pcap + p] = F[k];
    }
    if (P.has_sand) {
#pragma unroll
        for (int k = 0; k < 3; k++) buf.dps[(size_t)k * pcap + p] = dps[k];
    }
    if (P.has_force) {
        fdt[p] = 0.0f;
        fdt[(size_t)pcap + p] = 0.0f;
        fdt[2 * (size_t)pcap + p] = 0.0f;
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// Host launchers (declarations in slosh_api.hip).

static inline uint32_t div_up_t(uint64_t a, uint32_t b) { return (uint32_t)((a + b - 1) / b); }
static inline uint32_t min_t(uint32_t a, uint32_t b) { return a < b ? a : b; }

static inline PBuf to_pbuf(const ParticleBuffers &b) {
    PBuf p;
    p.pos = b.pos;
    p.vm = b.vm;
    p.C = b.C;
    p.F = b.F;
    p.vgd = b.vgd;
    p.ids = b.ids;
    p.dps = b.dps;
    return p;
}

// Workgroups of a per-block kernel (a multiple of the XCDs): one block
// per workgroup up to the tuned persistent width; workgroups loop over the
// device-side block count. The count is not known here: dense scenes have a block per
// 300 to 500 particles, so one per 256 leaves few workgroups without a block (an idle
// one costs 0.2 ns of dispatch: 16384 of them 2.8 us), and 2048 fill the chip when
// particles are sparse.
static uint32_t block_grid(const StepParams &P) {
    const uint32_t likely = P.n / 256u > 2048u ? P.n / 256u : 2048u;
    return (min_t(P.cap < likely ? P.cap : likely, P.block_wgs) + 7u) & ~7u;
}

// Workgroups of one item each (a multiple of the XCDs), looping beyond eight times the
// persistent width: every entry sequence is at most its block's candidates and listed
// movers (together at most 2 n entries), in 64s; dense scenes have an item per 55
// particles, sparse ones (42k blocks of 50) one per 40.
static uint32_t item_grid(const StepParams &P) {
    const uint64_t likely = P.n / 32u > 4096u ? P.n / 32u : 4096u, most = max_items(P.n, P.cap);
    return (min_t((uint32_t)(likely < most ? likely : most), 8u * P.block_wgs) + 7u) & ~7u;
}

static SortInputs sort_inputs(const TransferBuffers &t) {
    SortInputs in;
    in.rlist = t.rlist;
    in.rcnt = t.rcnt;
    in.prev_keys = t.prev_keys;
    in.arrive = t.arrive;
    in.prev_stay = t.prev_stay;
    in.blist = t.blist_out;
    in.num_blocks = t.num_blocks;
    in.nbr = t.nbr_out;
    in.blk_cnt = t.blk_cnt;
    in.bin = t.bin;
    in.rsum = t.rsum;
    in.rel = t.rel;
    in.rshift = t.rshift;
    return in;
}

static NextTable next_table(const NextTableBuffers &next) {
    NextTable nt;
    nt.keys = next.keys;
    nt.counters = next.counters;
    nt.arrive = next.arrive;
    nt.mlist = next.mlist;
    nt.ovf_slot = next.ovf_slot;
    nt.ovf_hid = next.ovf_hid;
    nt.rlist = next.rlist;
    nt.rcnt = next.rcnt;
    nt.rsum = next.rsum;
    nt.rshift = next.rshift;
    nt.prime = next.prime;
    return nt;
}

static Members members_of(const TransferBuffers &t) {
    Members M;
    M.fast = t.fast;
    M.blist = t.blist;
    M.bin = t.bin;
    M.mlist = t.mlist;
    M.ovf_slot = t.ovf_slot;
    M.ovf_hid = t.ovf_hid;
    M.perm = t.perm;
    M.blk_start = t.blk_start;
    M.blk_cnt = t.blk_cnt;
    M.counters = t.counters;
    return M;
}

hipError_t launch_p2g(const StepParams &P, const ParticleBuffers &pb, uint32_t pcap, const TransferBuffers &t,
                      const PassEvents *ev, hipStream_t stream) {
    // 512 by size (the comment at P2G_SUB_N).
    const bool by_size = P.p2g_chunk == 512u;
    const bool sub = by_size && P.n <= P2G_SUB_N;
    const uint32_t chunk = by_size && P.n > P2G_WIDE_N ? 384u : P.p2g_chunk;
    auto kern = t.fast ? (sub             ? k_p2g<512, true, 2>
                          : chunk == 192u ? k_p2g<192, true, 1>
                          : chunk == 256u ? k_p2g<256, true, 1>
                          : chunk == 384u ? k_p2g<384, true, 1>
                                          : k_p2g<512, true, 1>)
                       : (sub             ? k_p2g<512, false, 2>
                          : chunk == 192u ? k_p2g<192, false, 1>
                          : chunk == 256u ? k_p2g<256, false, 1>
                          : chunk == 384u ? k_p2g<384, false, 1>
                                          : k_p2g<512, false, 1>);
    P2gArgs args;
    args.P = P;
    args.pos = pb.pos;
    args.vm = pb.vm;
    args.C = pb.C;
    args.fdt = t.fdt;
    args.pcap = pcap;
    args.M = members_of(t);
    args.in = sort_inputs(t);
    args.keys = t.keys;
    args.tiles = t.tiles;
    args.cell_cnt = t.cell_cnt;
    launch_kernel(ev, kern, dim3(block_grid(P)), dim3(sub ? 384 : 192), 0, stream, args);
    return hipGetLastError();
}

hipError_t launch_grid_update(const StepParams &P, const TransferBuffers &t, const ColliderBuffers &c,
                              const NextTableBuffers &next, uint32_t mode, uint32_t do_update, const PassEvents *ev,
                              hipStream_t stream) {
    Colliders cs;
    cs.shapes = c.shapes;
    cs.poses = c.poses;
    cs.mats = c.mats;
    cs.count = c.count;
    cs.mesh_vtx = c.mesh_vtx;
    cs.mesh_idx = c.mesh_idx;
    cs.mesh_nodes = c.mesh_nodes;
    cs.mesh_leaves = c.mesh_leaves;
    cs.mesh_base = c.mesh_base;
    cs.mesh_search = c.mesh_base ? c.mesh_base + SLOSH_MAX_COLLIDERS : nullptr;
    cs.mesh_size = c.mesh_base ? (const float *)(c.mesh_base + 2 * SLOSH_MAX_COLLIDERS) : nullptr;
    ItemLists items;
    items.items = t.items;
    items.rsum = t.rsum;
    items.rel = t.rel;
    items.blk_start = t.blk_start;
    items.taken = t.taken;
    items.stay = t.stay;
    items.n_items = t.n_items;
    items.rshift = t.rshift;
    // Trimesh projection (a BVH walk) is compiled into its own instance so that
    // scenes without meshes keep the smaller kernel.
    launch_kernel(ev, c.mesh_vtx ? k_grid_update<true> : k_grid_update<false>, dim3(block_grid(P)),
                  dim3(c.mesh_vtx ? 64 * MESH_WAVES : 64), 0, stream, P,
                  (const float4 *)t.tiles, t.nodes, t.nbr, t.keys, cs, (const NodeColl *)t.coll_prev,
                  (NodeColl *)t.coll_cur, members_of(t), items, next_table(next), mode, do_update);
    return hipGetLastError();
}

hipError_t launch_pack_mesh(const float4 *vtx, const uint32_t *idx, uint32_t count, float4 *nodes, float4 *leaves,
                            hipStream_t stream) {
    hipLaunchKernelGGL(k_pack_mesh, dim3(div_up_t(count, 256)), dim3(256), 0, stream, vtx, idx, count, nodes, leaves);
    return hipGetLastError();
}

hipError_t launch_g2p_update(const StepParams &P, const ParticleBuffers &in, const ParticleBuffers &out,
                             const StaticBuffers &s, uint32_t pcap, const TransferBuffers &t,
                             const NextTableBuffers &next, const BodyBuffers &bb, const PassEvents *ev,
                             hipStream_t stream) {
    G2pArgs args;
    args.P = P;
    args.in = to_pbuf(in);
    args.out = to_pbuf(out);
    args.st.prop = s.prop;
    args.st.model = s.model;
    args.st.dp0 = s.dp0;
    args.st.dp1 = s.dp1;
    args.st.scene_rec = s.scene_rec;
    args.pcap = pcap;
    args.fdt = t.fdt;
    args.nt = next_table(next);
    args.ns.taken = t.taken;
    args.ns.stay = t.stay;
    args.ns.errors = t.errors;
    args.bodies.poses = bb.poses;
    args.bodies.vels = bb.vels;
    args.bodies.mprops = bb.mprops;
    args.bodies.local_com = bb.local_com;
    args.bodies.impulses = bb.impulses;
    args.bodies.count = bb.count;
    // The lightest instance that handles every material present: neo-Hookean
    // only (no SVD code), fixed-corotated and neo-Hookean, every material.
    const bool nh_only = (P.tag_mask & ~2u) == 0u;
    const bool elastic_only = (P.tag_mask & ~3u) == 0u;
    auto kern = nh_only        ? k_g2p_update<2u, false>
                : elastic_only ? (P.svd_f64 ? k_g2p_update<3u, true> : k_g2p_update<3u, false>)
                               : (P.svd_f64 ? k_g2p_update<15u, true> : k_g2p_update<15u, false>);
    // One more workgroup (the last) integrates the rigid bodies.
    launch_kernel(ev, kern, dim3(item_grid(P) + 1u), dim3(64), 0, stream, args, members_of(t),
                  (const uint32_t *)t.items, (const float4 *)t.nodes);
    return hipGetLastError();
}

hipError_t launch_g2p(const StepParams &P, const ParticleBuffers &b, uint32_t pcap, const TransferBuffers &t,
                      const PassEvents *ev, hipStream_t stream) {
    launch_kernel(ev, k_g2p, dim3(block_grid(P)), dim3(256), 0, stream, P, to_pbuf(b), pcap, t.perm, t.blist,
                  (const uint32_t *)t.blk_start, (const uint32_t *)t.blk_cnt, t.nbr, (const float4 *)t.nodes,
                  t.counters);
    return hipGetLastError();
}

hipError_t launch_particle_update(const StepParams &P, const ParticleBuffers &b, const StaticBuffers &s, uint32_t pcap,
                                  float *fdt, const PassEvents *ev, hipStream_t stream) {
    if (P.n == 0) return hipSuccess;
    PStatic st;
    st.prop = s.prop;
    st.model = s.model;
    st.dp0 = s.dp0;
    st.dp1 = s.dp1;
    st.scene_rec = s.scene_rec;
    auto kern = P.tag_mask == 2u ? k_particle_update<2u, false>
                                 : (P.svd_f64 ? k_particle_update<15u, true> : k_particle_update<15u, false>);
    launch_kernel(ev, kern, dim3(div_up_t(P.n, 256)), dim3(256), 0, stream, P, to_pbuf(b), st, pcap, fdt);
    return hipGetLastError();
}

// For each run of equal scene ids among slots [slot0, slot0 + n): the by-id
// records of the run's first particle into its scene's table entry.
__global__ __launch_bounds__(256) void k_scene_records(const float4 *__restrict__ pos, const uint32_t *__restrict__ ids,
                                                       uint32_t slot0, uint32_t n, PStatic st,
                                                       float4 *__restrict__ scene_rec) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t scene = __float_as_uint(pos[slot0 + i].w) >> 1;
    if (i > 0 && (__float_as_uint(pos[slot0 + i - 1].w) >> 1) == scene) return;
    const uint32_t oid = ids[slot0 + i];
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    scene_rec[4 * (size_t)scene] = st.prop[oid];
    scene_rec[4 * (size_t)scene + 1] = st.model[oid];
    scene_rec[4 * (size_t)scene + 2] = st.dp0 ? st.dp0[oid] : zero;
    scene_rec[4 * (size_t)scene + 3] = st.dp1 ? st.dp1[oid] : zero;
}

// Then each scene's mass, the largest particle mass of its uploaded particles
// (the enabled ones share it, the disabled ones have +0), into the unused third
// component of its plastic record (zeroed by k_scene_records). As unsigned bits,
// non-negative floats order as their values. An upload holds each scene's
// particles in one run, so a wave almost always covers one scene: it reduces
// first and sends one atomic (per-particle atomics on one address per scene
// serialize in L2: 11.4M of them on 256 records took ~10 ms).
__global__ __launch_bounds__(256) void k_scene_mass(const float4 *__restrict__ pos, const float4 *__restrict__ vm,
                                                    uint32_t slot0, uint32_t n, float4 *__restrict__ scene_rec) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    const uint32_t scene = valid ? __float_as_uint(pos[slot0 + i].w) >> 1 : SLOSH_NONE;
    const uint32_t m = valid ? __float_as_uint(vm[slot0 + i].w) : 0u;
    // Lane 0 holds the wave's first index, so it is valid whenever any lane is.
    const uint32_t s0 = (uint32_t)__shfl((int)scene, 0);
    if (__ballot(valid && scene != s0) == 0ull) {
        uint32_t x = m;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x = max(x, (uint32_t)__shfl_xor((int)x, o));
        if (lane_id() == 0 && s0 != SLOSH_NONE) atomicMax((uint32_t *)&scene_rec[4 * (size_t)s0 + 3].z, x);
    } else if (valid) {
        atomicMax((uint32_t *)&scene_rec[4 * (size_t)scene + 3].z, m);
    }
}

hipError_t launch_scene_records(const float4 *pos, const float4 *vm, const uint32_t *ids, uint32_t slot0, uint32_t n,
                                const StaticBuffers &s, float4 *scene_rec, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    PStatic st;
    st.prop = s.prop;
    st.model = s.model;
    st.dp0 = s.dp0;
    st.dp1 = s.dp1;
    st.scene_rec = nullptr;
    hipLaunchKernelGGL(k_scene_records, dim3(div_up_t(n, 256)), dim3(256), 0, stream, pos, ids, slot0, n, st,
                       scene_rec);
    hipLaunchKernelGGL(k_scene_mass, dim3(div_up_t(n, 256)), dim3(256), 0, stream, pos, vm, slot0, n, scene_rec);
    return hipGetLastError();
}

hipError_t launch_timestep_bound(const StepParams &P, const ParticleBuffers &b, const StaticBuffers &s, uint32_t pcap,
                                 uint32_t *out, hipStream_t stream) {
    if (P.n == 0) return hipSuccess;
    PStatic st;
    st.prop = s.prop;
    st.model = s.model;
    st.dp0 = s.dp0;
    st.dp1 = s.dp1;
    st.scene_rec = s.scene_rec;
    hipLaunchKernelGGL(k_timestep_bound, dim3(min_t(div_up_t(P.n, 256), 4096)), dim3(256), 0, stream, P, to_pbuf(b),
                       st, pcap, out);
    return hipGetLastError();
}

hipError_t launch_timestep_bound_partials(const StepParams &P, const ParticleBuffers &b, const StaticBuffers &s,
                                          uint32_t pcap, uint32_t *partials, uint32_t *out, hipStream_t stream) {
    PStatic st;
    st.prop = s.prop;
    st.model = s.model;
    st.dp0 = s.dp0;
    st.dp1 = s.dp1;
    st.scene_rec = s.scene_rec;
    const uint32_t groups = div_up_t(P.n, TSB_CHUNK);
    if (groups > 0)
        hipLaunchKernelGGL(k_timestep_bound_partials, dim3(groups), dim3(256), 0, stream, P, to_pbuf(b), st, pcap,
                           partials);
    hipLaunchKernelGGL(k_min_partials, dim3(1), dim3(256), 0, stream, partials, groups, out);
    return hipGetLastError();
}

hipError_t launch_rigid_update(const StepParams &P, const BodyBuffers &bb, const PassEvents *ev, hipStream_t stream) {
    if (bb.count == 0) return hipSuccess;
    Bodies b;
    b.poses = bb.poses;
    b.vels = bb.vels;
    b.mprops = bb.mprops;
    b.local_com = bb.local_com;
    b.impulses = bb.impulses;
    b.count = bb.count;
    launch_kernel(ev, k_rigid_update, dim3(1), dim3(64), 0, stream, P, b);
    return hipGetLastError();
}
