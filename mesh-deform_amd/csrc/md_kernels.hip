// HIP kernels of the ARAP path for CDNA4 (gfx950): cotan assembly, local step, rotated-edge
// right-hand side with FP64 residual, level-scheduled block-LDL^T sweeps, ARAP energy.
//
// Every kernel works on a LaunchSet (one or many meshes); the mesh of a block is found by a
// binary search of the block index in the launch's prefix table, so a single mesh, a static
// batch and a served mix of meshes all run through the same launches.
#define MD_KERNELS_DEVICE 1
#include "md_kernels.h"
#include "md_analysis.h"
#include "md_arap.h"

#include <cmath>
#include <string>
#include <type_traits>

namespace md {

namespace {

__device__ __forceinline__ int find_mesh(const LaunchSet &L, int b) {
    if (L.bmesh) return L.bmesh[b];
    int lo = 0, hi = L.nactive - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (L.prefix[mid] <= b) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Reciprocal, square root and reciprocal square root of the local step's Jacobi rotations:
// single hardware instructions in FP32 (about 1 ulp; the rotation is renormalised at the
// end), correctly rounded in FP64.
// (host builds of the rotation code, for the host diagnostic md_host_best_rotation, use the
// correctly rounded operations)
template <typename T> __host__ __device__ __forceinline__ T jrcp(T x);
template <> __host__ __device__ __forceinline__ float jrcp<float>(float x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}
template <> __host__ __device__ __forceinline__ double jrcp<double>(double x) { return 1.0 / x; }
template <typename T> __host__ __device__ __forceinline__ T jsqrt(T x);
template <> __host__ __device__ __forceinline__ float jsqrt<float>(float x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_sqrtf(x);
#else
    return std::sqrt(x);
#endif
}
template <> __host__ __device__ __forceinline__ double jsqrt<double>(double x) { return sqrt(x); }
template <typename T> __host__ __device__ __forceinline__ T jrsqrt(T x);
template <> __host__ __device__ __forceinline__ float jrsqrt<float>(float x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_rsqf(x);
#else
    return 1.0f / std::sqrt(x);
#endif
}
template <> __host__ __device__ __forceinline__ double jrsqrt<double>(double x) { return 1.0 / sqrt(x); }

// std::max<Scalar>(a, b) = (a < b) ? b : a; arap.h:199-218 pass the clamp first, so NaN
// yields the clamp.
__device__ __forceinline__ double ref_max(double a, double b) { return (a < b) ? b : a; }

// ---- cotan weights (arap.h:182-239) -----------------------------------------------------

// One thread per face: the three clamped half-cotangents of arap.h:199-218, 225-227.
__global__ __launch_bounds__(kBlock) void k_cotan_face(LaunchSet L) {
#pragma clang fp contract(off)
    int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    int f = (blockIdx.x - L.prefix[k]) * kBlock + threadIdx.x;
    if (f >= M.F) return;
    int i0 = M.tri[3 * f], i1 = M.tri[3 * f + 1], i2 = M.tri[3 * f + 2];
    d4 v0 = M.p[i0], v1 = M.p[i1], v2 = M.p[i2];
    double dx, dy, dz;
    dx = v1.x - v0.x; dy = v1.y - v0.y; dz = v1.z - v0.z;
    double l0 = ref_max(1e-8, dx * dx + dy * dy + dz * dz);
    dx = v2.x - v1.x; dy = v2.y - v1.y; dz = v2.z - v1.z;
    double l1 = ref_max(1e-8, dx * dx + dy * dy + dz * dz);
    dx = v0.x - v2.x; dy = v0.y - v2.y; dz = v0.z - v2.z;
    double l2 = ref_max(1e-8, dx * dx + dy * dy + dz * dz);
    l0 = sqrt(l0); l1 = sqrt(l1); l2 = sqrt(l2);
    const double semip = 0.5 * (l0 + l1 + l2);
    const double area = ref_max(1e-8, sqrt(semip * (semip - l0) * (semip - l1) * (semip - l2)));
    const double denom = 1.0 / (4.0 * area);
    double cot0 = (-l0 * l0 + l1 * l1 + l2 * l2) * denom;
    double cot1 = (l0 * l0 - l1 * l1 + l2 * l2) * denom;
    double cot2 = (l0 * l0 + l1 * l1 - l2 * l2) * denom;
    M.fe_val[3 * f] = ref_max(1e-10, cot0) * 0.5;
    M.fe_val[3 * f + 1] = ref_max(1e-10, cot1) * 0.5;
    M.fe_val[3 * f + 2] = ref_max(1e-10, cot2) * 0.5;
}

// One workgroup per 64-vertex slice, its slots dealt to the wavefronts column by column, four in
// flight each: a slot sums its face-edge contributions in face order (setFromTriplets' duplicate
// sum, arap.h:224,238) and stores w_ij and the weighted rest edge a_ij = w_ij (p_i - p_j) in FP64 and
// FP32. With diag, the weights also pass through LDS to the first wavefront, which sums each free
// vertex' in slot order (L_ii, arap.h:332) and the largest into amax (bits of a non-negative double; one
// address for all slices takes 12 ns per atomic, 25 us on the 164k icosphere).
// Bound by round trips per slot (face list, values, neighbour), so a lane taking a vertex' slots one after
// another took 59 us on a UV sphere of 3,202 with poles of 80 neighbours, and 37 on the 164k
// icosphere; the diagonal was a launch of its own (6 and 32 us, one atomic per vertex).
// Now 29 and 34 us, 7 on a sphere of 642 (10 and 6 for the diagonal).
constexpr int kCotSlots = 8;  // slot columns per round of a workgroup
__global__ __launch_bounds__(kBlock) void k_cotan_slot(LaunchSet L, double *diag, unsigned long long *amax) {
    __shared__ double wsh[kCotSlots][kSlice];
    const int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    const int slice = blockIdx.x - L.prefix[k], lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int iv = slice * kSlice + lane;
    const int s0 = M.slice_ptr[slice], wd = M.slice_ptr[slice + 1] - s0;
    const d4 pi = M.p[iv < M.n ? iv : 0];
    double acc = 0.0;
    for (int q0 = 0; q0 < wd; q0 += kCotSlots) {
        constexpr int kWaves = kBlock / 64, kU = kCotSlots / kWaves;
        int j[kU], e0[kU], e1[kU], f0[kU], f1[kU];
        d4 pj[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int q = q0 + u * kWaves + wave;
            j[u] = e0[u] = e1[u] = 0;
            if (q < wd) {
                const long long g = (long long)(s0 + q) * kSlice + lane;
                j[u] = M.sell_col[g];
                e0[u] = M.slot_fe_ptr[g];
                e1[u] = M.slot_fe_ptr[g + 1];
            }
        }
        // the first two face edges of every slot (all of an ordinary one's) at once
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            f0[u] = e1[u] > e0[u] ? M.slot_fe[e0[u]] : -1;
            f1[u] = e1[u] > e0[u] + 1 ? M.slot_fe[e0[u] + 1] : -1;
            if (q0 + u * kWaves + wave < wd) pj[u] = M.p[j[u]];
        }
        double w[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const double a = f0[u] >= 0 ? M.fe_val[f0[u]] : 0.0, b = f1[u] >= 0 ? M.fe_val[f1[u]] : 0.0;
            w[u] = (0.0 + a) + b;
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int q = q0 + u * kWaves + wave;
            if (q >= wd) break;
            for (int e = e0[u] + 2; e < e1[u]; ++e) w[u] += M.fe_val[M.slot_fe[e]];
            double ax = w[u] * (pi.x - pj[u].x), ay = w[u] * (pi.y - pj[u].y), az = w[u] * (pi.z - pj[u].z);
            if (iv >= M.n) { w[u] = 0.0; ax = ay = az = 0.0; }
            wsh[q - q0][lane] = j[u] == iv ? 0.0 : w[u];
            const long long g = (long long)(s0 + q) * kSlice + lane;
            M.w64[g] = w[u];
            M.w32[g] = (float)w[u];
            M.a64[g] = ax; M.a64[M.slots + g] = ay; M.a64[2 * M.slots + g] = az;
            M.a32[g] = (float)ax; M.a32[M.slots + g] = (float)ay; M.a32[2 * M.slots + g] = (float)az;
        }
        if (!diag) continue;
        __syncthreads();
        if (wave == 0)
            for (int q = 0; q < min(kCotSlots, wd - q0); ++q) acc += wsh[q][lane];
        __syncthreads();
    }
    if (!diag || wave != 0) return;
    const bool free_row = iv < M.nf;
    if (free_row) diag[iv] = acc;
    unsigned long long top = free_row ? (unsigned long long)__double_as_longlong(fabs(acc)) : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = max(top, (unsigned long long)__shfl_xor(top, o));
    if (lane == 0) atomicMax(amax + slice % kFacMaxima * kFacMaxStride, top);
}

// Lane moves inside a row of 16 lanes (DPP control CTRL).
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int CTRL> __device__ __forceinline__ double dpp_move(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)u, CTRL, 0xF, 0xF, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// v + the value of the other row of each pair (Half: of the other half of the wavefront).
template <bool Half> __device__ __forceinline__ void rows_swap(unsigned u, unsigned (&o)[2]) {
    if constexpr (Half) {
        const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        o[0] = a[0]; o[1] = a[1];
    } else {
        const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        o[0] = a[0]; o[1] = a[1];
    }
}
template <bool Half> __device__ __forceinline__ float rows_sum(float v) {
    unsigned a[2];
    rows_swap<Half>(__builtin_bit_cast(unsigned, v), a);
    return __builtin_bit_cast(float, a[0]) + __builtin_bit_cast(float, a[1]);
}
template <bool Half> __device__ __forceinline__ double rows_sum(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    unsigned lo[2], hi[2];
    rows_swap<Half>((unsigned)u, lo);
    rows_swap<Half>((unsigned)(u >> 32), hi);
    return __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]) +
           __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
}
// Sum over the wavefront, in every lane (quads, half rows, rows, row pairs, halves).
template <typename T> __device__ __forceinline__ T wave_sum(T v) {
    v += dpp_move<0xB1>(v);
    v += dpp_move<0x4E>(v);
    v += dpp_move<0x141>(v);
    v += dpp_move<0x140>(v);
    v = rows_sum<false>(v);
    return rows_sum<true>(v);
}
// v of lane l (the same l in every lane).
__device__ __forceinline__ double lane_value(double v, int l) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), l);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// One-rings longer than kRingSlots: where at most kFewLong lanes of a wavefront have one (a pole among
// vertices of six neighbours), the wavefront takes their remaining slots together, a lane per slot, one
// long ring after another: a round trip and nine sums (about 1.2 us) each, where every eight slots of
// a ring are a round trip of the whole wavefront otherwise (the rotations of a UV sphere of 3,202 with poles
// of 80 neighbours: 16 -> 8 us).
constexpr int kRingSlots = 16, kFewLong = 4;
// Lanes whose one-ring (wd > kRingSlots slots from s0; vertex iv) goes on past kRingSlots.
__device__ __forceinline__ unsigned long long long_rings(const MD_G MeshDev &M, bool live, int iv, int s0) {
    return __ballot(live && M.sell_col[(long long)(s0 + kRingSlots) * kSlice + iv % kSlice] != iv);
}

// ---- local step (arap.h:354-384) ----------------------------------------------------------

// One Jacobi rotation of the symmetric 4x4 matrix a on the pair (P, Q); v accumulates the
// eigenvectors (columns).
template <typename T, int P, int Q>
__host__ __device__ __forceinline__ void jrot(T (&a)[4][4], T (&v)[4][4]) {
    T apq = a[P][Q];
    T scale = fabs(a[P][P]) + fabs(a[Q][Q]);
    if (!(fabs(apq) > (sizeof(T) == 4 ? T(1e-9) : T(1e-18)) * scale) ) {
        if (fabs(apq) <= (sizeof(T) == 4 ? T(1e-30) : T(1e-300))) return;
        if (scale > T(0)) return;
    }
    T theta = (a[Q][Q] - a[P][P]) * jrcp<T>(T(2) * apq);
    T t = (theta >= T(0) ? T(1) : T(-1)) * jrcp<T>(fabs(theta) + jsqrt<T>(theta * theta + T(1)));
    T c = jrsqrt<T>(t * t + T(1));
    T s = t * c;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (r == P || r == Q) continue;
        T arp = a[r][P], arq = a[r][Q];
        T np = c * arp - s * arq, nq = s * arp + c * arq;
        a[r][P] = np; a[P][r] = np;
        a[r][Q] = nq; a[Q][r] = nq;
    }
    a[P][P] = a[P][P] - t * apq;
    a[Q][Q] = a[Q][Q] + t * apq;
    a[P][Q] = T(0); a[Q][P] = T(0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        T vp = v[r][P], vq = v[r][Q];
        v[r][P] = c * vp - s * vq;
        v[r][Q] = s * vp + c * vq;
    }
}

// R = argmax_{R in SO(3)} tr(R M) for the covariance M = sum_j a_j e'_j^T, returned as the
// unit quaternion (x, y, z, w). This is the rotation V diag(1,1,det(V U^T)) U^T of the
// reference's JacobiSVD step (arap.h:376-382), computed as the dominant eigenvector of
// Horn's symmetric 4x4 matrix N (J. Opt. Soc. Am. A 4(4), 1987).
//
// best_rotation_jacobi: cyclic Jacobi sweeps that start from the basis of the previous
// rotation (p = previous quaternion): the left-multiplication matrix L(p) is orthogonal with
// first column p, so L^T N L is already nearly diagonal when the rotation changed little and
// one or two sweeps converge. The converged eigenvector does not depend on the start.
template <typename T>
__host__ __device__ __forceinline__ void best_rotation_jacobi(const T (&m)[9], T px, T py, T pz, T pw, T &qx, T &qy,
                                                              T &qz, T &qw) {
    const T Sxx = m[0], Sxy = m[1], Sxz = m[2], Syx = m[3], Syy = m[4], Syz = m[5], Szx = m[6],
            Szy = m[7], Szz = m[8];
    const T N[4][4] = {{Sxx + Syy + Szz, Syz - Szy, Szx - Sxz, Sxy - Syx},
                       {Syz - Szy, Sxx - Syy - Szz, Sxy + Syx, Szx + Sxz},
                       {Szx - Sxz, Sxy + Syx, -Sxx + Syy - Szz, Syz + Szy},
                       {Sxy - Syx, Szx + Sxz, Syz + Szy, -Sxx - Syy + Szz}};
    {
        T pn = px * px + py * py + pz * pz + pw * pw;
        T inv = jrsqrt<T>(pn > T(0) ? pn : T(1));
        if (!(pn > T(0))) { px = 0; py = 0; pz = 0; pw = 1; }
        px *= inv; py *= inv; pz *= inv; pw *= inv;
    }
    // L(p) for p = (w, x, y, z) in the (scalar, vector) order of N's rows
    T v[4][4] = {{pw, -px, -py, -pz}, {px, pw, -pz, py}, {py, pz, pw, -px}, {pz, -py, px, pw}};
    T a[4][4];
    {
        T t[4][4];  // t = N L
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) t[r][c] = N[r][0] * v[0][c] + N[r][1] * v[1][c] + N[r][2] * v[2][c] + N[r][3] * v[3][c];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = r; c < 4; ++c) {
                T x = v[0][r] * t[0][c] + v[1][r] * t[1][c] + v[2][r] * t[2][c] + v[3][r] * t[3][c];
                a[r][c] = x;
                a[c][r] = x;
            }
    }
    constexpr int kSweeps = sizeof(T) == 4 ? 6 : 10;
    for (int sw = 0; sw < kSweeps; ++sw) {
        T off = fabs(a[0][1]) + fabs(a[0][2]) + fabs(a[0][3]) + fabs(a[1][2]) + fabs(a[1][3]) + fabs(a[2][3]);
        T dia = fabs(a[0][0]) + fabs(a[1][1]) + fabs(a[2][2]) + fabs(a[3][3]);
        if (!(off > (sizeof(T) == 4 ? T(1e-8) : T(1e-17)) * dia)) break;
        jrot<T, 0, 1>(a, v); jrot<T, 0, 2>(a, v); jrot<T, 0, 3>(a, v);
        jrot<T, 1, 2>(a, v); jrot<T, 1, 3>(a, v); jrot<T, 2, 3>(a, v);
    }
    // column of the largest eigenvalue, by selects (an index into v would put v in scratch)
    T best = a[0][0];
    T q0 = v[0][0], q1 = v[1][0], q2 = v[2][0], q3 = v[3][0];
#pragma unroll
    for (int c = 1; c < 4; ++c) {
        const bool b = a[c][c] > best;
        best = b ? a[c][c] : best;
        q0 = b ? v[0][c] : q0;
        q1 = b ? v[1][c] : q1;
        q2 = b ? v[2][c] : q2;
        q3 = b ? v[3][c] : q3;
    }
    T nrm = jrsqrt<T>(q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3);
    // canonical sign: scalar part >= 0
    if (q0 < T(0)) nrm = -nrm;
    qw = q0 * nrm; qx = q1 * nrm; qy = q2 * nrm; qz = q3 * nrm;
}

// Cofactor (-1)^(I+J) det(a without row I and column J) of a 4x4 matrix (indices fixed at
// compile time, so a stays in registers).
template <typename T, int I, int J>
__host__ __device__ __forceinline__ T cofactor(const T (&a)[4][4]) {
    constexpr int r0 = I == 0 ? 1 : 0, r1 = I <= 1 ? 2 : 1, r2 = I <= 2 ? 3 : 2;
    constexpr int k0 = J == 0 ? 1 : 0, k1 = J <= 1 ? 2 : 1, k2 = J <= 2 ? 3 : 2;
    const T d = a[r0][k0] * (a[r1][k1] * a[r2][k2] - a[r1][k2] * a[r2][k1]) -
                a[r0][k1] * (a[r1][k0] * a[r2][k2] - a[r1][k2] * a[r2][k0]) +
                a[r0][k2] * (a[r1][k0] * a[r2][k1] - a[r1][k1] * a[r2][k0]);
    return ((I + J) & 1) ? -d : d;
}

// Column col of adj(a) for a symmetric 4x4 a.
template <typename T>
__host__ __device__ __forceinline__ void adj_column(const T (&a)[4][4], int col, T &v0, T &v1, T &v2, T &v3) {
    if (col == 0) {
        v0 = cofactor<T, 0, 0>(a); v1 = cofactor<T, 1, 0>(a); v2 = cofactor<T, 2, 0>(a); v3 = cofactor<T, 3, 0>(a);
    } else if (col == 1) {
        v0 = cofactor<T, 0, 1>(a); v1 = cofactor<T, 1, 1>(a); v2 = cofactor<T, 2, 1>(a); v3 = cofactor<T, 3, 1>(a);
    } else if (col == 2) {
        v0 = cofactor<T, 0, 2>(a); v1 = cofactor<T, 1, 2>(a); v2 = cofactor<T, 2, 2>(a); v3 = cofactor<T, 3, 2>(a);
    } else {
        v0 = cofactor<T, 0, 3>(a); v1 = cofactor<T, 1, 3>(a); v2 = cofactor<T, 2, 3>(a); v3 = cofactor<T, 3, 3>(a);
    }
}

// best_rotation: the largest eigenvalue lambda of N by Newton's method on its characteristic
// polynomial P(x) = x^4 + c2 x^2 + c1 x + c0 with c2 = -2 |M|_F^2, c1 = -8 det M, c0 = det N
// (N is traceless; Theobald, Acta Cryst. A61 (2005) 478-480, "quaternion characteristic
// polynomial"), started at sqrt(3/2 |c2|) = sqrt(3) |M|_F, an upper bound of lambda (the sum
// of M's singular values), from where Newton's iterates decrease monotonically to the largest
// root of a polynomial with real roots. The eigenvector is then the largest column of
// adj(N - lambda I) = prod_{j>1}(lambda_j - lambda) v v^T, taken at its largest diagonal entry.
// When that entry is small against |N|^3 the top eigenvalue is (nearly) repeated -- a rank-1
// or reflection-ambiguous covariance -- the adjugate loses accuracy, and the warm-started
// Jacobi sweeps decide instead. A zero covariance keeps the previous rotation.
// The rotation does not depend on the covariance's scale, but the products on the way to it do, up to its
// seventh power (FP32: past about 1e5 or below 1e-5 they leave the range): m is first scaled, exactly, by the
// power of two that brings its largest entry into [0.5, 1).
template <typename T>
__host__ __device__ __forceinline__ bool best_rotation(const T (&cov)[9], T px, T py, T pz, T pw, T &qx, T &qy, T &qz,
                                                       T &qw) {
    T big = fabs(cov[0]);
#pragma unroll
    for (int i = 1; i < 9; ++i) big = fmax(big, fabs(cov[i]));
    int e;
    (void)frexp(big, &e);
    T m[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) m[i] = ldexp(cov[i], -e);
    const T Sxx = m[0], Sxy = m[1], Sxz = m[2], Syx = m[3], Syy = m[4], Syz = m[5], Szx = m[6],
            Szy = m[7], Szz = m[8];
    const T f2 = Sxx * Sxx + Sxy * Sxy + Sxz * Sxz + Syx * Syx + Syy * Syy + Syz * Syz + Szx * Szx + Szy * Szy +
                 Szz * Szz;
    const T n00 = Sxx + Syy + Szz, n01 = Syz - Szy, n02 = Szx - Sxz, n03 = Sxy - Syx;
    const T n11 = Sxx - Syy - Szz, n12 = Sxy + Syx, n13 = Szx + Sxz;
    const T n22 = -Sxx + Syy - Szz, n23 = Syz + Szy;
    const T n33 = -Sxx - Syy + Szz;
    const T c2 = T(-2) * f2;
    const T c1 = T(-8) * (Sxx * (Syy * Szz - Syz * Szy) - Sxy * (Syx * Szz - Syz * Szx) + Sxz * (Syx * Szy - Syy * Szx));
    // det N from the 2x2 minors of rows (0, 1) and rows (2, 3)
    const T s0 = n00 * n11 - n01 * n01, s1 = n00 * n12 - n01 * n02, s2 = n00 * n13 - n01 * n03;
    const T s3 = n01 * n12 - n11 * n02, s4 = n01 * n13 - n11 * n03, s5 = n02 * n13 - n12 * n03;
    const T t5 = n22 * n33 - n23 * n23, t4 = n12 * n33 - n13 * n23, t3 = n12 * n23 - n13 * n22;
    const T t2 = n02 * n33 - n03 * n23, t1 = n02 * n23 - n03 * n22, t0 = n02 * n13 - n03 * n12;
    const T c0 = s0 * t5 - s1 * t4 + s2 * t3 + s3 * t2 - s4 * t1 + s5 * t0;
    if (!(f2 > T(0))) {  // no edges carry weight: keep the previous rotation
        T pn = px * px + py * py + pz * pz + pw * pw;
        T inv = jrsqrt<T>(pn > T(0) ? pn : T(1));
        if (!(pn > T(0))) { px = 0; py = 0; pz = 0; pw = 1; inv = 1; }
        if (pw < T(0)) inv = -inv;
        qx = px * inv; qy = py * inv; qz = pz * inv; qw = pw * inv;
        return true;
    }
    const T scale = jsqrt<T>(T(1.5) * (-c2));
    T lam = scale;
    constexpr T kTol = sizeof(T) == 4 ? T(1e-6) : T(1e-14);
    for (int it = 0; it < 60; ++it) {
        const T l2 = lam * lam;
        const T p = (l2 + c2) * l2 + c1 * lam + c0;
        const T dp = T(4) * l2 * lam + T(2) * c2 * lam + c1;
        if (!(dp > T(0))) break;  // at (or beyond) a multiple root: the fallback decides
        const T step = p / dp;
        lam -= step;
        if (!(fabs(step) > kTol * scale)) break;
    }
    // a = N - lambda I; the diagonal of adj(a) (principal 3x3 minors) picks the column
    const T a[4][4] = {{n00 - lam, n01, n02, n03},
                       {n01, n11 - lam, n12, n13},
                       {n02, n12, n22 - lam, n23},
                       {n03, n13, n23, n33 - lam}};
    const T d0 = cofactor<T, 0, 0>(a), d1 = cofactor<T, 1, 1>(a), d2 = cofactor<T, 2, 2>(a),
            d3 = cofactor<T, 3, 3>(a);
    T best = fabs(d0);
    int col = 0;
    if (fabs(d1) > best) { best = fabs(d1); col = 1; }
    if (fabs(d2) > best) { best = fabs(d2); col = 2; }
    if (fabs(d3) > best) { best = fabs(d3); col = 3; }
    constexpr T kGap = sizeof(T) == 4 ? T(1e-2) : T(1e-4);
    if (!(best > kGap * scale * scale * scale)) {
        best_rotation_jacobi<T>(m, px, py, pz, pw, qx, qy, qz, qw);
        return false;
    }
    // column `col` of adj(a) (a is symmetric, so adj(a) is too); then once more at the
    // Rayleigh quotient of that vector, whose error is the square of the vector's: the rounding
    // of det N moves the polynomial's root by up to eps |N|^4 / prod(gaps), and the vector's
    // error is that shift over the gap
    T v0, v1, v2, v3;
    adj_column<T>(a, col, v0, v1, v2, v3);
    {
        const T nv = v0 * v0 + v1 * v1 + v2 * v2 + v3 * v3;
        const T w0 = n00 * v0 + n01 * v1 + n02 * v2 + n03 * v3, w1 = n01 * v0 + n11 * v1 + n12 * v2 + n13 * v3;
        const T w2 = n02 * v0 + n12 * v1 + n22 * v2 + n23 * v3, w3 = n03 * v0 + n13 * v1 + n23 * v2 + n33 * v3;
        const T rq = (v0 * w0 + v1 * w1 + v2 * w2 + v3 * w3) / nv;
        const T b[4][4] = {{n00 - rq, n01, n02, n03},
                           {n01, n11 - rq, n12, n13},
                           {n02, n12, n22 - rq, n23},
                           {n03, n13, n23, n33 - rq}};
        adj_column<T>(b, col, v0, v1, v2, v3);
    }
    T nrm = jrsqrt<T>(v0 * v0 + v1 * v1 + v2 * v2 + v3 * v3);
    if (v0 < T(0)) nrm = -nrm;  // canonical sign: scalar part >= 0
    qw = v0 * nrm; qx = v1 * nrm; qy = v2 * nrm; qz = v3 * nrm;
    return true;
}

template <typename T>
__host__ __device__ __forceinline__ void quat_to_mat(T qx, T qy, T qz, T qw, T (&R)[9]) {
    T s = T(2) / (qx * qx + qy * qy + qz * qz + qw * qw);
    R[0] = T(1) - s * (qy * qy + qz * qz); R[1] = s * (qx * qy - qw * qz); R[2] = s * (qx * qz + qw * qy);
    R[3] = s * (qx * qy + qw * qz); R[4] = T(1) - s * (qx * qx + qz * qz); R[5] = s * (qy * qz - qw * qx);
    R[6] = s * (qx * qz - qw * qy); R[7] = s * (qy * qz + qw * qx); R[8] = T(1) - s * (qx * qx + qy * qy);
}

template <typename T> __device__ __forceinline__ const T *aplanes(const MD_G MeshDev &M);
template <> __device__ __forceinline__ const float *aplanes<float>(const MD_G MeshDev &M) { return M.a32; }
template <> __device__ __forceinline__ const double *aplanes<double>(const MD_G MeshDev &M) { return M.a64; }

// One lane per vertex (all n, constrained ones too, as arap.h:358 loops over every vertex):
// covariance sum_j w_ij (p_i - p_j)(p'_i - p'_j)^T (arap.h:366-374) from the slice's slots,
// then the rotation. The deformed edge p'_i - p'_j is formed in FP64 and rounded to T.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_local(LaunchSet L) {
    using V = typename V4T<T>::type;
    int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    int slice = (blockIdx.x - L.prefix[k]) * kSlicesPerBlock + (threadIdx.x >> 6);
    int lane = threadIdx.x & 63;
    if (slice >= M.nslices) return;
    const int iv = min(slice * kSlice + lane, M.n - 1);  // (the last slice's spare lanes help with long rings)
    const bool live = slice * kSlice + lane < M.n;
    const T *A = aplanes<T>(M);
    int s0 = M.slice_ptr[slice], wd = M.slice_ptr[slice + 1] - s0;
    const d4 pi = M.pp[iv];
    const V prev = reinterpret_cast<const V *>(M.quat)[iv];  // (early: its latency is hidden)
    T c[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    auto add = [&](T (&o)[9], T ax, T ay, T az, T ex, T ey, T ez) {
        o[0] += ax * ex; o[1] += ax * ey; o[2] += ax * ez;
        o[3] += ay * ex; o[4] += ay * ey; o[5] += ay * ez;
        o[6] += az * ex; o[7] += az * ey; o[8] += az * ez;
    };
    // 8 slots at a time: ids and edges first, then the neighbour gathers, then arithmetic
    // (slots past the slice width are clamped; they are padding with zero edges anyway)
    constexpr int kU = 8;
    unsigned long long far = wd > kRingSlots ? long_rings(M, live, iv, s0) : 0;
    if (__popcll(far) > kFewLong) far = 0;
    for (int q0 = 0, end = far ? kRingSlots : wd; q0 < end; q0 += kU) {
        int jj[kU];
        T ex_[kU], ey_[kU], ez_[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            long long g = (long long)(s0 + min(q0 + u, wd - 1)) * kSlice + lane;
            jj[u] = M.sell_col[g];
            bool ok = q0 + u < wd;
            ex_[u] = ok ? A[g] : T(0);
            ey_[u] = ok ? A[M.slots + g] : T(0);
            ez_[u] = ok ? A[2 * M.slots + g] : T(0);
        }
        d4 pj[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) pj[u] = M.pp[jj[u]];
#pragma unroll
        for (int u = 0; u < kU; ++u)
            add(c, ex_[u], ey_[u], ez_[u], (T)(pi.x - pj[u].x), (T)(pi.y - pj[u].y), (T)(pi.z - pj[u].z));
    }
    for (; far; far &= far - 1) {
        const int l = __ffsll(far) - 1;
        const double px = lane_value(pi.x, l), py = lane_value(pi.y, l), pz = lane_value(pi.z, l);
        T o[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        for (int q = kRingSlots + lane; q < wd; q += 64) {
            const long long g = (long long)(s0 + q) * kSlice + l;
            const d4 pj = M.pp[M.sell_col[g]];
            add(o, A[g], A[M.slots + g], A[2 * M.slots + g], (T)(px - pj.x), (T)(py - pj.y), (T)(pz - pj.z));
        }
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            const T sum = wave_sum(o[e]);
            if (lane == l) c[e] += sum;
        }
    }
    if (!live) return;
    T qx, qy, qz, qw;
    best_rotation<T>(c, prev.x, prev.y, prev.z, prev.w, qx, qy, qz, qw);
    V out;
    out.x = qx; out.y = qy; out.z = qz; out.w = qw;
    reinterpret_cast<V *>(M.quat)[iv] = out;
}

// ---- right-hand side and residual (arap.h:393-414) --------------------------------------

// One lane per free vertex i:
//   r_i = sum_j [ 1/2 (R_i + R_j) a_ij  -  w_ij (p'_i - p'_j) ]
// over all neighbours j. With p'_j equal to the targets for constrained j this is
// b_i - (L p')_i for the reference's b = bFixed + sum_j w_ij/2 (R_i + R_j)(p_i - p_j)
// (arap.h:395-414) and L of arap.h:325-332, so the solve returns the correction to p'.
// The rotation term is in T, the weight term in FP64.
// r_i of one free vertex, slots kU at a time (ids and edges, then the neighbour gathers).
template <typename T, int kU>
__device__ __forceinline__ typename V4T<T>::type residual_of(const MD_G MeshDev &M, int iv) {
    using V = typename V4T<T>::type;
    const int slice = iv / kSlice, lane = iv % kSlice;
    const T *A = aplanes<T>(M);
    const V *Q = reinterpret_cast<const V *>(M.quat);
    int s0 = M.slice_ptr[slice], wd = M.slice_ptr[slice + 1] - s0;
    d4 pi = M.pp[iv];
    V qi = Q[iv];
    T sax = 0, say = 0, saz = 0;   // sum_j a_ij
    T rx = 0, ry = 0, rz = 0;      // sum_j R_j a_ij
    double lx = 0, ly = 0, lz = 0; // sum_j w_ij (p'_i - p'_j)
    for (int q0 = 0; q0 < wd; q0 += kU) {
        int jj[kU];
        T ax_[kU], ay_[kU], az_[kU];
        double w_[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            long long g = (long long)(s0 + min(q0 + u, wd - 1)) * kSlice + lane;
            jj[u] = M.sell_col[g];
            bool ok = q0 + u < wd;
            ax_[u] = ok ? A[g] : T(0);
            ay_[u] = ok ? A[M.slots + g] : T(0);
            az_[u] = ok ? A[2 * M.slots + g] : T(0);
            w_[u] = ok ? M.w64[g] : 0.0;
        }
        V qj_[kU];
        d4 pj_[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) { qj_[u] = Q[jj[u]]; pj_[u] = M.pp[jj[u]]; }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            T ax = ax_[u], ay = ay_[u], az = az_[u];
            T Rj[9];
            quat_to_mat<T>(qj_[u].x, qj_[u].y, qj_[u].z, qj_[u].w, Rj);
            sax += ax; say += ay; saz += az;
            rx += Rj[0] * ax + Rj[1] * ay + Rj[2] * az;
            ry += Rj[3] * ax + Rj[4] * ay + Rj[5] * az;
            rz += Rj[6] * ax + Rj[7] * ay + Rj[8] * az;
            double w = w_[u];
            lx += w * (pi.x - pj_[u].x); ly += w * (pi.y - pj_[u].y); lz += w * (pi.z - pj_[u].z);
        }
    }
    T Ri[9];
    quat_to_mat<T>(qi.x, qi.y, qi.z, qi.w, Ri);
    T bx = T(0.5) * (Ri[0] * sax + Ri[1] * say + Ri[2] * saz + rx);
    T by = T(0.5) * (Ri[3] * sax + Ri[4] * say + Ri[5] * saz + ry);
    T bz = T(0.5) * (Ri[6] * sax + Ri[7] * say + Ri[8] * saz + rz);
    V out;
    out.x = (T)((double)bx - lx);
    out.y = (T)((double)by - ly);
    out.z = (T)((double)bz - lz);
    out.w = 0;
    return out;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_residual(LaunchSet L) {
    using V = typename V4T<T>::type;
    int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    int slice = (blockIdx.x - L.prefix[k]) * kSlicesPerBlock + (threadIdx.x >> 6);
    int lane = threadIdx.x & 63;
    if (slice >= M.nslices_free) return;
    int iv = slice * kSlice + lane;
    if (iv >= M.nf) return;
    reinterpret_cast<V *>(M.r)[iv] = residual_of<T, 8>(M, iv);
}

// ---- block LDL^T sweeps (arap.h:416-429) --------------------------------------------------

template <typename T> __device__ __forceinline__ const T *tptr(const void *p) {
    return reinterpret_cast<const T *>(p);
}

// Sum of cnt partial vectors U[k * stride + e], k = 0 .. cnt-1, in that order. One partial is
// one load; more are loaded 8 at a time (clamped addresses, masked values) so their
// latencies overlap.
constexpr int kPartialBatch = 8;
// The same in the panel-preloading tiles (few waves: registers to spare), so the 9-16 partials
// of a wide owner's x, or the 9-16 update slots of a wide front's position, arrive in one round.
constexpr int kWidePartialBatch = 16;
// Level launches of at most this many tiles load their panel entries ahead of the vector
// (latency-bound: few waves); larger ones keep the register count low for occupancy.
constexpr int kPreloadMaxTiles = 2048;

template <typename V, int B = kPartialBatch>
__device__ __forceinline__ V sum_partials(const V *U, int cnt, int stride, int e) {
    using T = decltype(V{}.x);
    if (cnt == 1) return U[e];
    V a;
    a.x = 0; a.y = 0; a.z = 0; a.w = 0;
    for (int k0 = 0; k0 < cnt; k0 += B) {
        V b[B];
#pragma unroll
        for (int u = 0; u < B; ++u) b[u] = U[(long long)min(k0 + u, cnt - 1) * stride + e];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            T m = (k0 + u < cnt) ? T(1) : T(0);
            a.x += m * b[u].x; a.y += m * b[u].y; a.z += m * b[u].z;
        }
    }
    return a;
}

// Children's partial updates at position pos of a level front: the sum of its uk slots (slot k
// at k * m + pos; the children's partials fill them in child order, unused ones are zero), so
// their addresses follow from the tile alone.
template <typename V, int B = kPartialBatch>
__device__ __forceinline__ V pull_slots(const MD_G MeshDev &M, const SnDev &S, int pos) {
    return sum_partials<V, B>(reinterpret_cast<const V *>(M.upart) + S.ubase, S.uk, S.w + S.noff, pos);
}

// The update-slot sums of two front positions (a: ona lanes, b: onb lanes), their loads
// issued together, B slots of each per round: the first column tile of a forward tile needs
// both its columns' and its off rows' sums, and one round trip instead of two brings them. The
// sums run in slot order, as pull_slots' do (inactive lanes read position 0 and add nothing).
template <typename V, int B>
__device__ __forceinline__ void pull_slots_pair(const MD_G MeshDev &M, const SnDev &S, int pa, bool ona, int pb,
                                                bool onb, V &a, V &b) {
    using T = decltype(V{}.x);
    const MD_G V *U = reinterpret_cast<const MD_G V *>(M.upart) + S.ubase;
    const int cnt = S.uk, stride = S.w + S.noff;
    const int ea = ona ? pa : 0, eb = onb ? pb : 0;
    a.x = 0; a.y = 0; a.z = 0; a.w = 0;
    b = a;
    if (cnt == 1) {
        const V ua = U[ea], ub = U[eb];
        if (ona) a = ua;
        if (onb) b = ub;
        return;
    }
    for (int k0 = 0; k0 < cnt; k0 += B) {
        V ua[B], ub[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const long long row = (long long)min(k0 + u, cnt - 1) * stride;
            ua[u] = U[row + ea];
            ub[u] = U[row + eb];
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const T m = (k0 + u < cnt) ? T(1) : T(0);
            const T ma = ona ? m : T(0), mb = onb ? m : T(0);
            a.x += ma * ua[u].x; a.y += ma * ua[u].y; a.z += ma * ua[u].z;
            b.x += mb * ub[u].x; b.y += mb * ub[u].y; b.z += mb * ub[u].z;
        }
    }
}

// g[i] = P[min(i, n - 1) * stride] for i < N (n >= 1): a column of a panel tile loaded into
// registers ahead of the vector it multiplies; entries past n are valid panel values that meet
// zero vector entries.
template <int N, typename T>
__device__ __forceinline__ void panel_load(const T *P, long long stride, int n, T *g) {
#pragma unroll
    for (int i = 0; i < N; ++i) g[i] = P[(long long)min(i, n - 1) * stride];
}

// acc += sum_{i < N} g[i] * v[i] (v[i] = 0 for i >= n).
template <int N, typename T, typename V>
__device__ __forceinline__ void panel_dot(const T *g, const V *v, T &ax, T &ay, T &az) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const V x = v[i];
        ax += g[i] * x.x; ay += g[i] * x.y; az += g[i] * x.z;
    }
}

// acc += sum_{i < n} P[i * stride] * v[i] for n <= N (N = 16, 32 or 64): all N loads are
// issued together (addresses clamped to [0, n-1], or to 0 when n <= 0; values masked), so
// P[0] and v[0] must be readable.
template <int N, typename T, typename V>
__device__ __forceinline__ void tile_dot(const T *P, long long stride, const V *v, int n, T &ax, T &ay, T &az) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        int ii = max(0, min(i, n - 1));
        T g = P[(long long)ii * stride];
        g = i < n ? g : T(0);
        V x = v[ii];
        ax += g * x.x; ay += g * x.y; az += g * x.z;
    }
}

template <typename T, typename V>
__device__ __forceinline__ void tile_dot_any(const T *P, long long stride, const V *v, int n, T &ax, T &ay, T &az) {
    if (n <= 16) tile_dot<16>(P, stride, v, n, ax, ay, az);
    else if (n <= 32) tile_dot<32>(P, stride, v, n, ax, ay, az);
    else tile_dot<64>(P, stride, v, n, ax, ay, az);
}

// Forward tile (s, r0, q0), one wavefront:
//   v_d[q0 .. q0+64) = r[c0 + q] + children's updates landing on those columns,
//   v_o[r0 .. r0+64) = children's updates landing on those off rows (first column tile),
//   z_s[q0 ..] = v_d (first row tile),
//   partial q0/64 of u_s on rows [r0, r0+64) = (q0 == 0 ? v_o : 0) - G_s[rows, cols] v_d.
// Children's updates arrive as kc partial vectors; each lane pulls the contributions listed
// for its position (host-built lists in child order), so no two lanes write the same place.
// fwd_tile loads the tile's G entries (N = 16, 32 or 64 columns) while the contributions arrive:
// a shorter chain of dependent loads for twice the registers (launches of few tiles);
// fwd_tile_lean loads them after the contributions.
template <int N, typename T>
__device__ __forceinline__ void fwd_tile(const MD_G MeshDev &M, const SnDev &S, int r0, int q0, int qn, int rn) {
    using V = typename V4T<T>::type;
    __shared__ V vd[kTile];
    __shared__ V vo[kTile];
    const int lane = threadIdx.x, w = S.w, no = S.noff, kcb = q0 / kTile;
    const V *R = reinterpret_cast<const V *>(M.r);
    V b, o;
    b.x = 0; b.y = 0; b.z = 0; b.w = 0;
    o = b;
    if (lane < qn) b = R[S.c0 + q0 + lane];
    // column-major G_s: entry (row r, column q) at q * no + r
    T g[N];
    if (rn > 0) panel_load<N, T>(tptr<T>(M.pc) + S.pc_off + (long long)q0 * no + r0 + min(lane, rn - 1), no, qn, g);
    const long long dst = lane < rn ? M.udst[S.roff + r0 + lane] : 0;  // this row's slot in the parent
    if (kcb == 0) {
        // columns and off rows: their slots in one round trip
        V c;
        pull_slots_pair<V, kPartialBatch>(M, S, q0 + lane, lane < qn, w + r0 + lane, lane < rn, c, o);
        if (lane < qn) { b.x += c.x; b.y += c.y; b.z += c.z; b.w = 0; }
    } else if (lane < qn) {
        const V c = pull_slots<V, kWidePartialBatch>(M, S, q0 + lane);
        b.x += c.x; b.y += c.y; b.z += c.z; b.w = 0;
    }
    vd[lane] = b;
    vo[lane] = o;
    __syncthreads();
    if (r0 == 0 && lane < qn) reinterpret_cast<V *>(M.z)[S.c0 + q0 + lane] = vd[lane];
    if (rn == 0) return;
    T ax = 0, ay = 0, az = 0;
    panel_dot<N, T, V>(g, vd, ax, ay, az);
    if (lane < rn) {
        V out;
        out.x = (kcb == 0 ? o.x : T(0)) - ax;
        out.y = (kcb == 0 ? o.y : T(0)) - ay;
        out.z = (kcb == 0 ? o.z : T(0)) - az;
        out.w = 0;
        reinterpret_cast<V *>(M.upart)[dst + (long long)kcb * S.dstride] = out;
    }
}

template <typename T>
__device__ __forceinline__ void fwd_tile_lean(const MD_G MeshDev &M, const SnDev &S, int r0, int q0, int qn, int rn) {
    using V = typename V4T<T>::type;
    __shared__ V vd[kTile];
    __shared__ V vo[kTile];
    const int lane = threadIdx.x, w = S.w, no = S.noff, kcb = q0 / kTile;
    const V *R = reinterpret_cast<const V *>(M.r);
    {
        V b;
        b.x = 0; b.y = 0; b.z = 0; b.w = 0;
        if (lane < qn) {
            b = R[S.c0 + q0 + lane];
            V c = pull_slots<V>(M, S, q0 + lane);
            b.x += c.x; b.y += c.y; b.z += c.z; b.w = 0;
        }
        vd[lane] = b;
        V o;
        o.x = 0; o.y = 0; o.z = 0; o.w = 0;
        if (kcb == 0 && lane < rn) o = pull_slots<V>(M, S, w + r0 + lane);
        vo[lane] = o;
    }
    __syncthreads();
    if (r0 == 0 && lane < qn) reinterpret_cast<V *>(M.z)[S.c0 + q0 + lane] = vd[lane];
    if (rn == 0) return;
    const T *G = tptr<T>(M.pc) + S.pc_off + (long long)q0 * no + r0 + min(lane, rn - 1);
    T ax = 0, ay = 0, az = 0;
    tile_dot_any<T, V>(G, no, vd, qn, ax, ay, az);
    if (lane < rn) {
        V o = vo[lane], out;
        out.x = (kcb == 0 ? o.x : T(0)) - ax;
        out.y = (kcb == 0 ? o.y : T(0)) - ay;
        out.z = (kcb == 0 ? o.z : T(0)) - az;
        out.w = 0;
        reinterpret_cast<V *>(M.upart)[M.udst[S.roff + r0 + lane] + (long long)kcb * S.dstride] = out;
    }
}

template <typename T, bool Pre>
__global__ __launch_bounds__(kTile) void k_fwd(LaunchSet L, int level) {
    const int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    const TileDev tl = L.tiles ? L.tiles[blockIdx.x] : M.ftile[L.tbase[k] + (blockIdx.x - L.prefix[k])];
    const SnDev &S = tl.s;
    const int r0 = tl.a, q0 = tl.b;
    const int qn = min(kTile, S.w - q0), rn = max(0, min(kTile, S.noff - r0));
    if (!Pre) fwd_tile_lean<T>(M, S, r0, q0, qn, rn);
    else if (qn <= 16) fwd_tile<16, T>(M, S, r0, q0, qn, rn);
    else if (qn <= 32) fwd_tile<32, T>(M, S, r0, q0, qn, rn);
    else fwd_tile<64, T>(M, S, r0, q0, qn, rn);
}

// Backward tile (s, q0, p0), one wavefront: partial p0/64 of x_s on columns [q0, q0+64):
//   sum over rows p in [p0, p0+64) of [Dinv_s; G_s][p, q] * t[p],  t = [z_s; -x_off],
// read from the row-major copy (lanes on consecutive columns). x at off rows is the sum of
// the owner's partials (xloc gives where they are). bwd_tile loads the tile's panel rows (N =
// 16, 32 or 64) while t is gathered; bwd_tile_lean loads them afterwards.
template <int N, typename T>
__device__ __forceinline__ void bwd_tile(const MD_G MeshDev &M, const SnDev &S, int q0, int p0, int qn, int pn) {
    using V = typename V4T<T>::type;
    __shared__ V tv[kTile];
    const int lane = threadIdx.x, w = S.w;
    const V *X = reinterpret_cast<const V *>(M.xpart);
    const int p = p0 + lane;
    // a root (no off rows) has no forward tile: its right-hand side and children's
    // contributions are gathered here (z = r + contributions, as the forward tile forms it)
    const bool root = S.noff == 0;
    V t;
    t.x = 0; t.y = 0; t.z = 0; t.w = 0;
    int4 xl = make_int4(0, 0, 0, 0);
    if (lane < pn) {
        if (p >= w) xl = M.xloc[S.roff + p - w];
        else if (root) t = reinterpret_cast<const V *>(M.r)[S.c0 + p];
        else t = reinterpret_cast<const V *>(M.z)[S.c0 + p];
    }
    T g[N];
    panel_load<N, T>(tptr<T>(M.pr) + S.pr_off + (long long)p0 * w + q0 + min(lane, qn - 1), w, pn, g);
    if (lane < pn && p >= w) {
        const V a = sum_partials<V, kWidePartialBatch>(X + xl.x, xl.z, xl.y, 0);
        t.x = -a.x; t.y = -a.y; t.z = -a.z;
    }
    if (lane < pn && p < w && root) {
        const V c = pull_slots<V, kWidePartialBatch>(M, S, p);
        t.x += c.x; t.y += c.y; t.z += c.z;
    }
    t.w = 0;
    tv[lane] = t;
    __syncthreads();
    T ax = 0, ay = 0, az = 0;
    panel_dot<N, T, V>(g, tv, ax, ay, az);
    if (lane < qn) {
        V out;
        out.x = ax; out.y = ay; out.z = az; out.w = 0;
        reinterpret_cast<V *>(M.xpart)[S.xoff + (long long)(p0 / kTile) * w + q0 + lane] = out;
    }
}

template <typename T>
__device__ __forceinline__ void bwd_tile_lean(const MD_G MeshDev &M, const SnDev &S, int q0, int p0, int qn, int pn) {
    using V = typename V4T<T>::type;
    __shared__ V tv[kTile];
    const int lane = threadIdx.x, w = S.w;
    const V *X = reinterpret_cast<const V *>(M.xpart);
    {
        V t;
        t.x = 0; t.y = 0; t.z = 0;
        int p = p0 + lane;
        if (lane < pn) {
            if (p < w && S.noff == 0) {  // a root: no forward tile (as in bwd_tile)
                t = reinterpret_cast<const V *>(M.r)[S.c0 + p];
                const V c = pull_slots<V>(M, S, p);
                t.x += c.x; t.y += c.y; t.z += c.z;
            } else if (p < w) {
                t = reinterpret_cast<const V *>(M.z)[S.c0 + p];
            } else {
                int4 xl = M.xloc[S.roff + p - w];
                V a = sum_partials<V>(X + xl.x, xl.z, xl.y, 0);
                t.x = -a.x; t.y = -a.y; t.z = -a.z;
            }
        }
        t.w = 0;
        tv[lane] = t;
    }
    __syncthreads();
    const T *P = tptr<T>(M.pr) + S.pr_off + (long long)p0 * w + q0 + min(lane, qn - 1);
    T ax = 0, ay = 0, az = 0;
    tile_dot_any<T, V>(P, w, tv, pn, ax, ay, az);
    if (lane < qn) {
        V out;
        out.x = ax; out.y = ay; out.z = az; out.w = 0;
        reinterpret_cast<V *>(M.xpart)[S.xoff + (long long)(p0 / kTile) * w + q0 + lane] = out;
    }
}

template <typename T, bool Pre>
__global__ __launch_bounds__(kTile) void k_bwd(LaunchSet L, int level) {
    const int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    const TileDev tl = L.tiles ? L.tiles[blockIdx.x] : M.btile[L.tbase[k] + (blockIdx.x - L.prefix[k])];
    const SnDev &S = tl.s;
    const int q0 = tl.a, p0 = tl.b;
    const int qn = min(kTile, S.w - q0), pn = min(kTile, S.w + S.noff - p0);
    if (!Pre) bwd_tile_lean<T>(M, S, q0, p0, qn, pn);
    else if (pn <= 16) bwd_tile<16, T>(M, S, q0, p0, qn, pn);
    else if (pn <= 32) bwd_tile<32, T>(M, S, q0, p0, qn, pn);
    else bwd_tile<64, T>(M, S, q0, p0, qn, pn);
}

// Record of one supernode of a bottom subtree (16 ints, as the host lays it out).
struct SubNode {
    int c0, w, noff, fb;     // columns, off rows, forward front base in LDS
    int pc, pr, cp, ob;      // G offset, [Dinv; G] offset, contribution entries, off-row sources
    int uo, xo, xs, pa;      // root: first update-slot entry (udst) or -1; x output, LDS column base
                             //   of x, position prefix (host emulation only)
    int pb, pq, pad0, pad1;  // off-row prefix, column prefix (within the height)
};

// Last record j in [a, b) whose prefix (field F) is <= t.
template <int SubNode::*F>
__device__ __forceinline__ int sub_find(const SubNode *N, int a, int b, int t) {
    int lo = a, hi = b - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (N[mid].*F <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// One subtree as the host lays it out: records [sub.x, sub.y), height table offset sub.z, sub.w
// heights; rows [row.x, +row.y); forward positions [row.z, +row.w), backward off rows [ext.x, +ext.y).
struct SubTree {
    int4 sub, row;
    int2 ext;
};
__device__ __forceinline__ SubTree sub_tree(const MD_G MeshDev &M, int k) {
    const int4 e = M.srow[2 * k + 1];
    return SubTree{M.sub[k], M.srow[2 * k], make_int2(e.x, e.y)};
}

// Panel entries of a sweep item kept in registers, loaded while the positions before it are formed
// (their addresses depend on the layout alone).
constexpr int kSubAhead = 16;

// Bottom subtree, forward sweep, one workgroup per subtree, heights bottom-up with every front in LDS
// (position t of the subtree at F[t], its records' fronts one after another):
//   F = residual on the rows, else 0; per height
//   positions: F[t] += the children's update entries (none at height 0),
//   off rows:  F[w + i] -= G_s[i, 0..w) F[0 .. w)  (u_s in place; the root also stores u_s for its
//              parent outside the subtree);
// z = F on the rows at the end. Index lists are in LDS from the start and the next height's panel
// entries are loaded ahead, so a height costs no round trip of its own.
// With Fused (one-mesh launches), the residual is formed here: subtree rows straight into
// their front positions, level rows by blocks past the subtrees (no k_residual launch; more
// registers, so batches keep the separate residual).
// Bound by its chain of heights where the subtrees are few (a 10k icosphere's 91 in FP32: 11 us with the
// residual, 18 with one wavefront per subtree and dependent loads in every height), by occupancy
// where they are many.
template <typename T, bool Fused, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_sub_fwd(LaunchSet L, SubLds D) {
    using V = typename V4T<T>::type;
    extern __shared__ __align__(32) unsigned char sub_smem[];
    V *F = reinterpret_cast<V *>(sub_smem);
    SubNode *N = reinterpret_cast<SubNode *>(F + D.fwd);
    int2 *cp = reinterpret_cast<int2 *>(N + D.nodes);
    int *H = reinterpret_cast<int *>(cp + D.fwd);
    const int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    const int tid = threadIdx.x;
    const int bk = blockIdx.x - L.prefix[k];
    if (Fused && bk >= M.nsub) {
        // blocks past the subtrees: the residual of BLOCK rows of level supernodes
        const int j = (bk - M.nsub) * BLOCK + tid;
        if (j < M.nlrows) {
            const int i = M.lrows[j];
            reinterpret_cast<V *>(M.r)[i] = residual_of<T, 8>(M, i);
        }
        return;
    }
    const SubTree S = sub_tree(M, bk);
    const V *R = reinterpret_cast<const V *>(M.r);
    V *Z = reinterpret_cast<V *>(M.z);
    V *U = reinterpret_cast<V *>(M.upart);
    const T *G = tptr<T>(M.pc);
    {
        int4 *dst = reinterpret_cast<int4 *>(N);
        for (int i = tid; i < 4 * (S.sub.y - S.sub.x); i += BLOCK) dst[i] = M.snode[4 * S.sub.x + i];
        for (int i = tid; i <= S.sub.w; i += BLOCK) H[i] = M.sub_h[S.sub.z + i] - S.sub.x;
        V zero;
        zero.x = 0; zero.y = 0; zero.z = 0; zero.w = 0;
        for (int i = tid; i < S.row.w; i += BLOCK) {
            cp[i] = M.scp[S.row.z + i];
            F[i] = zero;
        }
    }
    __syncthreads();
    for (int t = tid; t < S.row.y; t += BLOCK)
        F[M.sfi[S.row.x + t]] = Fused ? residual_of<T, 8>(M, S.row.x + t) : R[S.row.x + t];
    // off row t of height h: its record and the first kSubAhead entries of its row of G_s
    T g[kSubAhead];
    int item = 0;
    auto load = [&](int a, int b, int t) {
        item = sub_find<&SubNode::pb>(N, a, b, t);
        const SubNode &s = N[item];
        panel_load<kSubAhead, T>(G + s.pc + (t - s.pb), s.noff, s.w, g);
    };
    auto rows_of = [&](int h) { return N[H[h + 1] - 1].pb + N[H[h + 1] - 1].noff; };
    if (tid < rows_of(0)) load(H[0], H[1], tid);
    __syncthreads();
    for (int h = 0; h < S.sub.w; ++h) {
        const int a = H[h], b = H[h + 1];
        if (h > 0) {
            const int p0 = N[a].cp - S.row.z, p1 = N[b - 1].cp - S.row.z + N[b - 1].w + N[b - 1].noff;
            for (int t = p0 + tid; t < p1; t += BLOCK) {
                // children's update entries: two inline, the rest from a -1-terminated list
                const int2 e = cp[t];
                V v = F[t];
                if (e.x >= 0) {
                    const V u = F[e.x];
                    v.x += u.x; v.y += u.y; v.z += u.z;
                }
                if (e.y >= 0) {
                    const V u = F[e.y];
                    v.x += u.x; v.y += u.y; v.z += u.z;
                } else if (e.y <= -2) {
                    for (int c = -2 - e.y;; ++c) {
                        const int q = M.sfc[c];
                        if (q < 0) break;
                        const V u = F[q];
                        v.x += u.x; v.y += u.y; v.z += u.z;
                    }
                }
                F[t] = v;
            }
            __syncthreads();
        }
        const int nrow = rows_of(h);
        for (int t = tid; t < nrow; t += BLOCK) {
            if (t != tid) load(a, b, t);
            const SubNode &s = N[item];
            const int i = t - s.pb;
            const V *v = F + s.fb;
            T ax = 0, ay = 0, az = 0;
            // column-major G_s: entry (row i, column q) at q * noff + i
            for (int q0 = 0; q0 < s.w; q0 += kSubAhead) {
                if (q0 > 0) panel_load<kSubAhead, T>(G + s.pc + i + (long long)q0 * s.noff, s.noff, s.w - q0, g);
#pragma unroll
                for (int u0 = 0; u0 < kSubAhead; u0 += 4) {
                    if (q0 + u0 < s.w) {
#pragma unroll
                        for (int u = u0; u < u0 + 4; ++u) {
                            const V x = v[min(q0 + u, s.w - 1)];
                            const T e = q0 + u < s.w ? g[u] : T(0);
                            ax += e * x.x; ay += e * x.y; az += e * x.z;
                        }
                    }
                }
            }
            V o = F[s.fb + s.w + i];
            o.x -= ax; o.y -= ay; o.z -= az;
            F[s.fb + s.w + i] = o;
            if (s.uo >= 0) U[M.udst[s.uo + i]] = o;  // the root: into the parent's slot
        }
        if (h + 1 < S.sub.w && tid < rows_of(h + 1)) load(b, H[h + 2], tid);
        __syncthreads();
    }
    for (int t = tid; t < S.row.y; t += BLOCK) Z[S.row.x + t] = F[M.sfi[S.row.x + t]];
}

// Bottom subtree, backward sweep, one workgroup per subtree, heights top-down with the subtree's z and
// solution columns and the fronts' off rows in LDS (z at F[t], x at F[ncols + t], off row e at
// F[2 ncols + e]). Off rows outside the subtree are gathered once at the start (-x, the sum of their
// owner's partials); per height
//   off rows: -x of those inside, from LDS,
//   columns:  x_s[q] = sum_p [Dinv_s; G_s][p, q] t[p], t = [z_s; off rows], four lanes per column
//             (rows p = lane mod 4, joined by DPP: a front of up to 4 kAhead rows is one load of kAhead
//             entries per lane, made a height ahead).
// A 10k icosphere's 91 subtrees in FP32: 9.5 us; one wavefront per subtree, one lane per column and
// a round trip for the sources and one for the panel in every height took 19. The 164k icosphere's
// 2,825 in FP64: 31 us (50). A batch's 7,413 in FP32: 50 us (73), 59 with kSubAhead entries ahead and its
// registers.
template <typename T>
__device__ __forceinline__ T quad_sum(T v) {
    v += dpp_move<0xB1>(v);
    return v + dpp_move<0x4E>(v);
}
template <typename T, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_sub_bwd(LaunchSet L, SubLds D) {
    using V = typename V4T<T>::type;
    extern __shared__ __align__(32) unsigned char sub_smem[];
    V *F = reinterpret_cast<V *>(sub_smem);
    SubNode *N = reinterpret_cast<SubNode *>(F + D.bwd);
    int *src = reinterpret_cast<int *>(N + D.nodes);  // x column of an off row inside the subtree, else -1
    int *H = src + D.off;
    const int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    const int tid = threadIdx.x;
    const V *X = reinterpret_cast<const V *>(M.xpart);
    const int bk = blockIdx.x - L.prefix[k];
    if (bk >= M.nsub) {
        // blocks past the subtrees: p' += x for BLOCK rows of level supernodes (x summed from
        // the partials of the level sweeps)
        const int j = (bk - M.nsub) * BLOCK + tid;
        if (j < M.nlrows) {
            const int i = M.lrows[j];
            const int4 ri = M.rowinfo[i];
            const V a = sum_partials<V>(X + ri.x, ri.z, ri.y, 0);
            d4 pv = M.pp[i];
            pv.x += (double)a.x; pv.y += (double)a.y; pv.z += (double)a.z;
            M.pp[i] = pv;
        }
        return;
    }
    const SubTree S = sub_tree(M, bk);
    const T *P = tptr<T>(M.pr);
    const int nc = S.row.y;
    V *x = F + nc, *off = F + 2 * nc;
    {
        int4 *dst = reinterpret_cast<int4 *>(N);
        for (int i = tid; i < 4 * (S.sub.y - S.sub.x); i += BLOCK) dst[i] = M.snode[4 * S.sub.x + i];
        for (int i = tid; i <= S.sub.w; i += BLOCK) H[i] = M.sub_h[S.sub.z + i] - S.sub.x;
        const V *Zs = reinterpret_cast<const V *>(M.z);
        for (int t = tid; t < nc; t += BLOCK) F[t] = Zs[S.row.x + t];
        for (int e = tid; e < S.ext.y; e += BLOCK) {
            const int2 d = M.sbo[S.ext.x + e];
            src[e] = d.y < 0 ? d.x : -1;
            if (d.y >= 0) {
                const V u = sum_partials<V>(X + d.x, d.y >> 16, d.y & 0xffff, 0);
                V o;
                o.x = -u.x; o.y = -u.y; o.z = -u.z; o.w = 0;
                off[e] = o;
            }
        }
    }
    __syncthreads();
    // column t of height h: its record and the first entries of the lane's rows
    // (FP32 launches of many subtrees: fewer registers, seven wavefronts per SIMD instead of four)
    constexpr int kAhead = BLOCK == kSubBlock || sizeof(T) == 8 ? kSubAhead : kSubAhead / 2;
    const int part = tid & 3;
    T g[kAhead];
    int item = 0;
    auto rows4 = [&](const SubNode &s, int q, int p0) {  // rows p0 + part, + 4, ...
        const int m = s.w + s.noff;
        const T *p = P + s.pr + q;
#pragma unroll
        for (int u = 0; u < kAhead; ++u) g[u] = p[(long long)min(p0 + part + 4 * u, m - 1) * s.w];
    };
    auto load = [&](int a, int b, int t) {
        item = sub_find<&SubNode::pq>(N, a, b, t);
        rows4(N[item], t - N[item].pq, 0);
    };
    auto cols_of = [&](int h) { return N[H[h + 1] - 1].pq + N[H[h + 1] - 1].w; };
    const int t0 = tid >> 2;
    if (t0 < cols_of(S.sub.w - 1)) load(H[S.sub.w - 1], H[S.sub.w], t0);
    for (int h = S.sub.w - 1; h >= 0; --h) {
        const int a = H[h], b = H[h + 1];
        if (h < S.sub.w - 1) {
            const int e0 = N[a].ob - S.ext.x, e1 = N[b - 1].ob - S.ext.x + N[b - 1].noff;
            for (int e = e0 + tid; e < e1; e += BLOCK) {
                const int c = src[e];
                if (c >= 0) {
                    const V u = x[c];
                    V o;
                    o.x = -u.x; o.y = -u.y; o.z = -u.z; o.w = 0;
                    off[e] = o;
                }
            }
            __syncthreads();
        }
        const int ncol = cols_of(h);
        for (int t = t0; t < ncol; t += BLOCK / 4) {
            if (t != t0) load(a, b, t);
            const SubNode &s = N[item];
            const int q = t - s.pq, m = s.w + s.noff;
            const V *zs = F + s.xs, *os = off + (s.ob - S.ext.x) - s.w;
            T ax = 0, ay = 0, az = 0;
            // row-major [Dinv_s; G_s]: entry (row p, column q) at p * w + q
            for (int p0 = 0; p0 < m; p0 += 4 * kAhead) {
                if (p0 > 0) rows4(s, q, p0);
#pragma unroll
                for (int u0 = 0; u0 < kAhead; u0 += 4) {
                    if (p0 + 4 * u0 < m) {
#pragma unroll
                        for (int u = u0; u < u0 + 4; ++u) {
                            const int p = p0 + part + 4 * u, pc = min(p, m - 1);
                            const V v = *(pc < s.w ? zs + pc : os + pc);
                            const T e = p < m ? g[u] : T(0);
                            ax += e * v.x; ay += e * v.y; az += e * v.z;
                        }
                    }
                }
            }
            ax = quad_sum(ax); ay = quad_sum(ay); az = quad_sum(az);
            if (part == 0) {
                V o;
                o.x = ax; o.y = ay; o.z = az; o.w = 0;
                x[s.xs + q] = o;
            }
        }
        if (h > 0 && t0 < cols_of(h - 1)) load(H[h - 1], a, t0);
        __syncthreads();
    }
    // x of the subtree's rows is final and read by nothing outside the subtree: p' += x
    for (int t = tid; t < nc; t += BLOCK) {
        const V o = x[t];
        d4 pv = M.pp[S.row.x + t];
        pv.x += (double)o.x; pv.y += (double)o.y; pv.z += (double)o.z;
        M.pp[S.row.x + t] = pv;
    }
}

// ---- Jacobi-preconditioned CG on the correction system (alternative to the sweeps) -------
//
// Solves A d = r for the three coordinates at once (three independent CG recurrences, one
// per coordinate), A = L of arap.h:325-332 over the free vertices, M = diag(A). d starts at 0:
// the residual r = b - A p' already warm-starts from the previous iterate. Every block works
// on 256 consecutive free vertices; dot products are per-block partials that each block of
// the next kernel reduces in the same fixed order (deterministic, no atomics).

template <typename T> __device__ __forceinline__ const T *wts(const MD_G MeshDev &M);
template <> __device__ __forceinline__ const float *wts<float>(const MD_G MeshDev &M) { return M.w32; }
template <> __device__ __forceinline__ const double *wts<double>(const MD_G MeshDev &M) { return M.w64; }

// Six block sums, in every thread: a wavefront's by lane moves, the wavefronts' through LDS
// (two LDS trees of eight barriers each took 4 of a CG step's 11 us). red is written once
// per kernel.
template <typename T> __device__ __forceinline__ void block_sum6(T (&v)[6], T (*red)[6]) {
    constexpr int kWaves = kBlock / 64;
#pragma unroll
    for (int q = 0; q < 6; ++q) v[q] = wave_sum(v[q]);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int q = 0; q < 6; ++q) red[threadIdx.x >> 6][q] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        v[q] = red[0][q];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) v[q] += red[w][q];
    }
}
// A block's sums of (r, u) and (w, u) into pa[blk] and pb[blk].
template <typename T, typename V>
__device__ __forceinline__ void block_partial2(T (&v)[6], MD_G V *pa, MD_G V *pb, int blk, T (*red)[6]) {
    block_sum6(v, red);
    if (threadIdx.x == 0) {
        V va, vb;
        va.x = v[0]; va.y = v[1]; va.z = v[2]; va.w = 0;
        vb.x = v[3]; vb.y = v[4]; vb.z = v[5]; vb.w = 0;
        pa[blk] = va;
        pb[blk] = vb;
    }
}

// L_ii = sum of every neighbour weight (arap.h:332), once per factorisation.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pcg_diag(LaunchSet L) {
    int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    int slice = (blockIdx.x - L.prefix[k]) * kSlicesPerBlock + (threadIdx.x >> 6);
    int lane = threadIdx.x & 63;
    if (slice >= M.nslices_free) return;
    int iv = slice * kSlice + lane;
    if (iv >= M.nf) return;
    int s0 = M.slice_ptr[slice], wd = M.slice_ptr[slice + 1] - s0;
    double d = 0.0;
    for (int q = 0; q < wd; ++q) d += M.w64[(long long)(s0 + q) * kSlice + lane];
    reinterpret_cast<T *>(M.diag)[iv] = (T)d;
}

// Jacobi-PCG in the Chronopoulos-Gear form (Chronopoulos and Gear, J. Comput. Appl. Math. 25
// (1989) 153-168): with u = M^-1 r and w = A u, step i forms
//   p = u + beta p, s = w + beta s, x += alpha p, r -= alpha s, u = M^-1 r, w = A u,
//   gamma = (r, u), delta = (w, u),
// and the next step takes beta = gamma_new / gamma, alpha = gamma_new / (delta - beta gamma_new /
// alpha): one reduction, so one launch, per CG iteration. The new u of a neighbour is formed from
// its r, w and s of the previous step, which live in the other buffer of each pair (parity i),
// so no lane reads what another writes. Per coordinate, a solve whose gamma fell below
// tol^2 gamma_0 keeps alpha = 0 (its x and r stay).
template <typename V> struct CgVecs {
    MD_G V *r[2], *w[2], *s[2], *x, *p;  // [0]: the parity a step reads, [1]: the one it writes
};
template <typename V>
__device__ __forceinline__ CgVecs<V> cg_vecs(const MD_G MeshDev &M, int parity) {
    MD_G V *r = reinterpret_cast<MD_G V *>(M.r), *v = reinterpret_cast<MD_G V *>(M.cg_v);
    const long long nf = M.nf, o = parity ? nf : 0;
    return {{parity ? v : r, parity ? r : v}, {v + nf + o, v + 2 * nf - o}, {v + 3 * nf + o, v + 4 * nf - o},
            reinterpret_cast<MD_G V *>(M.cg_x), reinterpret_cast<MD_G V *>(M.cg_p)};
}

// x = p = s_0 = 0, u = M^-1 r, w_0 = A u, partials of (r, u) and (w, u) (parity 0). One lane
// per free vertex in slice order (block b: vertices [256 b, 256 b + 256)).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pcg_init(LaunchSet L) {
    using V = typename V4T<T>::type;
    __shared__ T red[kBlock / 64][6];
    const int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    const int blk = blockIdx.x - L.prefix[k];
    const int slice = blk * kSlicesPerBlock + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int iv = slice * kSlice + lane;
    const CgVecs<V> c = cg_vecs<V>(M, 0);
    const MD_G T *D = reinterpret_cast<const MD_G T *>(M.diag);
    T dots[6] = {0, 0, 0, 0, 0, 0};  // (r, u), (w, u)
    if (slice < M.nslices_free && iv < M.nf) {
        const T *W = wts<T>(M);
        const int s0 = M.slice_ptr[slice], wd = M.slice_ptr[slice + 1] - s0;
        const V r = c.r[0][iv];
        const T di = D[iv], rdi = T(1) / di;
        const T ux = r.x * rdi, uy = r.y * rdi, uz = r.z * rdi;
        T yx = di * ux, yy = di * uy, yz = di * uz;
        for (int q = 0; q < wd; ++q) {
            const long long g = (long long)(s0 + q) * kSlice + lane;
            const int j = M.sell_col[g];
            if (j != iv && j < M.nf) {
                const V rj = c.r[0][j];
                const T wq = W[g] / D[j];
                yx -= wq * rj.x; yy -= wq * rj.y; yz -= wq * rj.z;
            }
        }
        V z;
        z.x = 0; z.y = 0; z.z = 0; z.w = 0;
        V w;
        w.x = yx; w.y = yy; w.z = yz; w.w = 0;
        c.w[0][iv] = w;
        c.s[0][iv] = z;
        c.x[iv] = z;
        c.p[iv] = z;
        dots[0] = r.x * ux; dots[1] = r.y * uy; dots[2] = r.z * uz;
        dots[3] = yx * ux; dots[4] = yy * uy; dots[5] = yz * uz;
    }
    MD_G V *part = reinterpret_cast<MD_G V *>(M.cg_part);
    const int nb = M.nblk_free;
    block_partial2<T, V>(dots, part, part + nb, blk, red);
}

// Step i (parity c = i & 1): reads r, w, s and the partials of parity c, writes those of 1 - c.
// Bound by the chain of one launch (10k icosphere: 34 workgroups): everything a lane reads,
// kPcgAhead slots of its one-ring included, is on its way before the partials are summed.
// A step of the 10k icosphere in FP32 takes 7.8 us (11.4 with LDS trees and the loads behind them), of
// the 164k one 16.4 (21.3) in FP32 and 27 (32) in FP64; with 8 slots ahead in FP64 the registers leave one
// wavefront per SIMD and that took 33.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pcg_step(LaunchSet L, int step) {
    using V = typename V4T<T>::type;
    constexpr int kPcgAhead = sizeof(T) == 4 ? 8 : 4;
    __shared__ T red[2][kBlock / 64][6];
    const int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    const int blk = blockIdx.x - L.prefix[k];
    const int slice = __builtin_amdgcn_readfirstlane(blk * kSlicesPerBlock + (int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int iv = slice * kSlice + lane;
    const int c = step & 1, n = 1 - c;
    const CgVecs<V> v = cg_vecs<V>(M, c);
    const MD_G T *D = reinterpret_cast<const MD_G T *>(M.diag);
    MD_G V *part = reinterpret_cast<MD_G V *>(M.cg_part);
    const int nb = M.nblk_free;
    MD_G V *scal = part + 4 * nb;  // (gamma, alpha) of each parity, then the first gamma
    const V gp = scal[2 * c], ap = scal[2 * c + 1], gz = scal[4];
    T sum[6] = {0, 0, 0, 0, 0, 0};
    for (int b = threadIdx.x; b < nb; b += kBlock) {
        const V x = part[2 * c * nb + b], y = part[(2 * c + 1) * nb + b];
        sum[0] += x.x; sum[1] += x.y; sum[2] += x.z;
        sum[3] += y.x; sum[4] += y.y; sum[5] += y.z;
    }
    const bool live = slice < M.nslices_free && iv < M.nf;
    const T *W = wts<T>(M);
    const bool inside = slice < M.nslices_free;
    const int s0 = inside ? M.slice_ptr[slice] : 0, wd = inside ? M.slice_ptr[slice + 1] - s0 : 0;
    V r = {}, w = {}, so = {}, p = {}, x = {}, nr[kPcgAhead], nw[kPcgAhead], ns[kPcgAhead];
    T di = T(1), wq[kPcgAhead], nd[kPcgAhead];
#pragma unroll
    for (int q = 0; q < kPcgAhead; ++q) {
        nr[q] = nw[q] = ns[q] = V{};
        wq[q] = T(0);
        nd[q] = T(1);
    }
    if (live) {
        r = v.r[0][iv]; w = v.w[0][iv]; so = v.s[0][iv];
        p = v.p[iv]; x = v.x[iv];
        di = D[iv];
        if (wd > 0) {
            int nj[kPcgAhead];
#pragma unroll
            for (int q = 0; q < kPcgAhead; ++q) {
                const long long g = (long long)(s0 + min(q, wd - 1)) * kSlice + lane;
                nj[q] = M.sell_col[g];
                wq[q] = W[g];
            }
#pragma unroll
            for (int q = 0; q < kPcgAhead; ++q) {
                // padding, constrained neighbours and slots past the slice's count as zero
                if (q >= wd || nj[q] >= M.nf || nj[q] == iv) { nj[q] = iv; wq[q] = T(0); }
                nr[q] = v.r[0][nj[q]]; nw[q] = v.w[0][nj[q]]; ns[q] = v.s[0][nj[q]];
                nd[q] = D[nj[q]];
            }
        }
    }
    block_sum6(sum, red[0]);
    const T ga[3] = {sum[0], sum[1], sum[2]}, de[3] = {sum[3], sum[4], sum[5]};
    T al[3], be[3];
    const T gprev[3] = {gp.x, gp.y, gp.z}, aprev[3] = {ap.x, ap.y, ap.z};
    const T g0[3] = {step == 0 ? ga[0] : gz.x, step == 0 ? ga[1] : gz.y, step == 0 ? ga[2] : gz.z};
    for (int q = 0; q < 3; ++q) {
        const bool conv = (double)ga[q] <= M.pcg_tol2 * (double)g0[q];
        if (step == 0) {
            be[q] = T(0);
            al[q] = (!conv && de[q] != T(0)) ? ga[q] / de[q] : T(0);
        } else if (conv || aprev[q] == T(0) || gprev[q] == T(0)) {
            be[q] = T(0);
            al[q] = T(0);
        } else {
            be[q] = ga[q] / gprev[q];
            const T den = de[q] - be[q] * ga[q] / aprev[q];
            al[q] = den != T(0) ? ga[q] / den : T(0);
        }
    }
    if (blockIdx.x == L.prefix[k] && threadIdx.x == 0) {  // for the next step
        V g, a;
        g.x = ga[0]; g.y = ga[1]; g.z = ga[2]; g.w = 0;
        a.x = al[0]; a.y = al[1]; a.z = al[2]; a.w = 0;
        scal[2 * n] = g;
        scal[2 * n + 1] = a;
        if (step == 0) scal[4] = g;  // the first gamma, for the stopping test
    }
    T dots[6] = {0, 0, 0, 0, 0, 0};
    if (live) {
        const T rdi = T(1) / di;
        // p = u + beta p, s = w + beta s, x += alpha p, r -= alpha s
        p.x = r.x * rdi + be[0] * p.x; p.y = r.y * rdi + be[1] * p.y; p.z = r.z * rdi + be[2] * p.z;
        V sn;
        sn.x = w.x + be[0] * so.x; sn.y = w.y + be[1] * so.y; sn.z = w.z + be[2] * so.z; sn.w = 0;
        x.x += al[0] * p.x; x.y += al[1] * p.y; x.z += al[2] * p.z;
        V rn;
        rn.x = r.x - al[0] * sn.x; rn.y = r.y - al[1] * sn.y; rn.z = r.z - al[2] * sn.z; rn.w = 0;
        v.p[iv] = p;
        v.x[iv] = x;
        v.s[1][iv] = sn;
        v.r[1][iv] = rn;
        // w = A u with u = M^-1 r of the new r; a neighbour's new u from its previous r, w, s
        const T ux = rn.x * rdi, uy = rn.y * rdi, uz = rn.z * rdi;
        T yx = di * ux, yy = di * uy, yz = di * uz;
        auto slot = [&](T wj, const V &rj, const V &uj, const V &sj) {
            yx -= wj * (rj.x - al[0] * (uj.x + be[0] * sj.x));
            yy -= wj * (rj.y - al[1] * (uj.y + be[1] * sj.y));
            yz -= wj * (rj.z - al[2] * (uj.z + be[2] * sj.z));
        };
#pragma unroll
        for (int q = 0; q < kPcgAhead; ++q)
            if (q < wd) slot(wq[q] / nd[q], nr[q], nw[q], ns[q]);
        for (int q = kPcgAhead; q < wd; ++q) {
            const long long g = (long long)(s0 + q) * kSlice + lane;
            const int j = M.sell_col[g];
            if (j != iv && j < M.nf) slot(W[g] / D[j], v.r[0][j], v.w[0][j], v.s[0][j]);
        }
        V wn;
        wn.x = yx; wn.y = yy; wn.z = yz; wn.w = 0;
        v.w[1][iv] = wn;
        dots[0] = rn.x * ux; dots[1] = rn.y * uy; dots[2] = rn.z * uz;
        dots[3] = yx * ux; dots[4] = yy * uy; dots[5] = yz * uz;
    }
    block_partial2<T, V>(dots, part + 2 * n * nb, part + (2 * n + 1) * nb, blk, red[1]);
}

// p' += d for the free vertices.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pcg_apply(LaunchSet L) {
    using V = typename V4T<T>::type;
    int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    int i = (blockIdx.x - L.prefix[k]) * kBlock + threadIdx.x;
    if (i >= M.nf) return;
    V x = reinterpret_cast<const V *>(M.cg_x)[i];
    d4 pv = M.pp[i];
    pv.x += (double)x.x; pv.y += (double)x.y; pv.z += (double)x.z;
    M.pp[i] = pv;
}

// ---- vertex normals of the deformed mesh (for rendering clients) --------------------------

// Area-weighted face normal of every face from p' (cross product of two edges, unnormalised),
// three doubles per face into fn.
__global__ __launch_bounds__(kBlock) void k_face_normals(LaunchSet L, double *fn) {
    int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    int f = (blockIdx.x - L.prefix[k]) * kBlock + threadIdx.x;
    if (f >= M.F) return;
    d4 a = M.pp[M.tri[3 * f]], b = M.pp[M.tri[3 * f + 1]], c = M.pp[M.tri[3 * f + 2]];
    double ux = b.x - a.x, uy = b.y - a.y, uz = b.z - a.z;
    double vx = c.x - a.x, vy = c.y - a.y, vz = c.z - a.z;
    fn[3 * f] = uy * vz - uz * vy;
    fn[3 * f + 1] = uz * vx - ux * vz;
    fn[3 * f + 2] = ux * vy - uy * vx;
}

// Per vertex: every incident face appears on exactly two of its one-ring slots (the two face
// edges at the vertex), so half the sum over the slots' face lists is the sum of incident
// face normals; normalised (zero stays zero). Output in internal order, or packed in original order
// (orig: original id of each internal id).
__global__ __launch_bounds__(kBlock) void k_vertex_normals(LaunchSet L, const double *fn, d4 *out, double *packed,
                                                           const int *orig) {
    int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    int slice = (blockIdx.x - L.prefix[k]) * kSlicesPerBlock + (threadIdx.x >> 6);
    int lane = threadIdx.x & 63;
    if (slice >= M.nslices) return;
    int iv = slice * kSlice + lane;
    if (iv >= M.n) return;
    int s0 = M.slice_ptr[slice], wd = M.slice_ptr[slice + 1] - s0;
    double x = 0, y = 0, z = 0;
    for (int q = 0; q < wd; ++q) {
        long long g = (long long)(s0 + q) * kSlice + lane;
        for (int e = M.slot_fe_ptr[g]; e < M.slot_fe_ptr[g + 1]; ++e) {
            int f = M.slot_fe[e] / 3;
            x += fn[3 * f]; y += fn[3 * f + 1]; z += fn[3 * f + 2];
        }
    }
    double nrm = sqrt(x * x + y * y + z * z);
    double inv = nrm > 0.0 ? 1.0 / nrm : 0.0;
    if (packed) {
        double *o = packed + 3 * (size_t)orig[iv];
        o[0] = x * inv; o[1] = y * inv; o[2] = z * inv;
        return;
    }
    d4 o;
    o.x = x * inv; o.y = y * inv; o.z = z * inv; o.w = 0.0;
    out[iv] = o;
}

// Internal-order vectors (positions or normals) to the caller's packed xyz in original vertex
// order: dst[3 v + c] = x[internal[v]].c. One thread per original vertex: dst may be pinned host memory,
// whose writes then leave in order.
__global__ __launch_bounds__(kBlock) void k_pack_xyz(const d4 *x, const int *internal, int n, double *dst,
                                                     unsigned long long *stamp) {
    const int v = blockIdx.x * kBlock + threadIdx.x;
    if (v == 0 && stamp) *stamp = wall_clock64();
    if (v >= n) return;
    const d4 p = x[internal[v]];
    double *o = dst + 3 * (size_t)v;
    o[0] = p.x; o[1] = p.y; o[2] = p.z;
}

// The same for the results of several meshes, one launch (a launch per mesh is 8 us for the 10 a full
// server finishes at a boundary, beside the next iteration's launches). The entries may lie in
// pinned host memory; block b belongs to the last entry whose first block is not past it.
__global__ __launch_bounds__(kBlock) void k_pack_results(const PackEntry *e, int count) {
    int lo = 0, hi = count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (e[mid].block <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
    }
    const PackEntry E = e[lo];
    const int v = ((int)blockIdx.x - E.block) * kBlock + threadIdx.x;
    if (v >= E.n) return;
    const d4 p = E.x[E.internal[v]];
    MD_G double *o = E.dst + 3 * (size_t)v;
    o[0] = p.x; o[1] = p.y; o[2] = p.z;
}

// Device workspace of the entry points that allocate nothing (md_mesh_normals_noalloc): one
// array per GPU, set aside when the code object loads and held until the process ends. Host
// code reaches it only through the address hipGetSymbolAddress returns on each device (the
// array's name in host code is a host-side stand-in, not a device address).
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// ---- ARAP energy -------------------------------------------------------------------------

// E = sum_i sum_j w_ij |(p'_i - p'_j) - R_i (p_i - p_j)|^2 over all vertices, in FP64; one
// partial sum per block of 256 vertices, reduced in a fixed order.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_energy(LaunchSet L) {
    using V = typename V4T<T>::type;
    __shared__ double red[kBlock];
    int k = find_mesh(L, blockIdx.x);
    const MD_G MeshDev &M = L.meshes[k];
    int lb = blockIdx.x - L.prefix[k];
    int slice = lb * kSlicesPerBlock + (threadIdx.x >> 6);
    int lane = threadIdx.x & 63;
    int iv = slice * kSlice + lane;
    double e = 0.0;
    if (slice < M.nslices && iv < M.n) {
        int s0 = M.slice_ptr[slice], wd = M.slice_ptr[slice + 1] - s0;
        V qi = reinterpret_cast<const V *>(M.quat)[iv];
        double R[9];
        quat_to_mat<double>((double)qi.x, (double)qi.y, (double)qi.z, (double)qi.w, R);
        d4 pi = M.p[iv], ppi = M.pp[iv];
        for (int q = 0; q < wd; ++q) {
            long long g = (long long)(s0 + q) * kSlice + lane;
            int j = M.sell_col[g];
            double w = M.w64[g];
            d4 pj = M.p[j], ppj = M.pp[j];
            double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            double tx = (ppi.x - ppj.x) - (R[0] * dx + R[1] * dy + R[2] * dz);
            double ty = (ppi.y - ppj.y) - (R[3] * dx + R[4] * dy + R[5] * dz);
            double tz = (ppi.z - ppj.z) - (R[6] * dx + R[7] * dy + R[8] * dz);
            e += w * (tx * tx + ty * ty + tz * tz);
        }
    }
    red[threadIdx.x] = e;
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) M.energy_part[lb] = red[0];
}

// The caller's packed xyz (original order, read in order: it may be pinned host memory) into
// internal order: p[iv] (may be null), and pp[iv] (may be null) the same for free vertices, the constrained
// ones (iv >= nf) taking their targets tgt[iv - nf] instead; with pp, identity rotations (arap.h:246-249).
// The first block clears `clear` (kFacWords) and thread 0 writes the clock to `stamp` (each may be null).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_unpack_xyz(UnpackArgs a) {
    using V = typename V4T<T>::type;
    const int v = blockIdx.x * kBlock + threadIdx.x;
    if (a.clear && blockIdx.x == 0)
        for (int i = v; i < kFacWords; i += kBlock) a.clear[i] = 0;
    if (v == 0 && a.stamp) *a.stamp = wall_clock64();
    if (v >= a.n) return;
    const int iv = a.internal[v];
    const double *s = a.xyz + 3 * (size_t)v;
    d4 x{s[0], s[1], s[2], 0.0};
    if (a.p) a.p[iv] = x;
    if (a.pp) {
        if (iv >= a.nf) {
            const double *t = a.tgt + 3 * (size_t)(iv - a.nf);
            x = d4{t[0], t[1], t[2], 0.0};
        }
        a.pp[iv] = x;
        V q;
        q.x = 0; q.y = 0; q.z = 0; q.w = 1;
        reinterpret_cast<V *>(a.quat)[iv] = q;
    }
}

// The clock and the factorization's flag (if any) to the host, between two phases' launches.
__global__ void k_publish(unsigned long long *stamp, const int *flag, int *out) {
    *stamp = wall_clock64();
    if (flag) *out = *flag;
}

// Targets of several meshes: entry t writes its position into the p' entry at its address.
__global__ __launch_bounds__(kBlock) void k_scatter_entries(const TargetEntry *e, int k) {
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= k) return;
    const TargetEntry x = e[t];
    *reinterpret_cast<MD_G d4 *>(x.addr) = d4{x.x, x.y, x.z, 0.0};
}

// ---- numeric factorization (arap.h:337, SimplicialLDLT::compute) ------------------------
// Multifrontal block LDL^T in FP64, one height of the supernodal tree at a time, each front by as many
// workgroups as it has parts or tiles (small fronts by one). Every supernode's front lives in its own
// workspace blocks; the children's update matrices are added in child order, so the factor is
// deterministic.

constexpr int kFacBlock = 256;

// Least pivot: 1e-14 of the largest diagonal entry.
__device__ __forceinline__ double pivot_floor(const FacArgs &A) {
    unsigned long long m = 0;
#pragma unroll
    for (int i = 0; i < kFacMaxima; ++i) m = max(m, A.amax[i * kFacMaxStride]);
    return 1e-14 * __longlong_as_double((long long)m);
}

constexpr int kFb = 64;  // columns of a pivot block swept at a time


// The first w columns of a front during the sweeps: step s reads one of two workspaces (P, all rows m
// apart; T, pivot rows w apart, with S, off rows noff apart; column-major) and writes the other, so no
// workgroup overwrites what another still reads. Block (s, s) of the workspace that step s reads holds
// A_ss^{-1} (the inverse is formed where the block is completed). The front's other columns, the update
// matrix, are updated in place.
struct FrontBuf {
    MD_G double *d, *f;  // pivot rows, off rows
    long long ldd, ldf;
};
__device__ __forceinline__ FrontBuf front_buf(const FacArgs &A, const FacDev &S, int s) {
    if (s & 1) return FrontBuf{A.T + S.toff, A.S + S.soff, S.w, S.noff};
    return FrontBuf{A.P + S.poff, A.P + S.poff + S.w, S.m, S.m};
}

// Front of each supernode of one height: its first w columns and the update matrix, lower part: for
// each entry the original one (L_jj and -w_ij for free i > j), then
// the children's update entries in child order. A gather: the children's row maps are inverted in LDS
// (front row -> row of the child, -1 where it has none), every entry is summed by one lane in a
// register and written once, so there is no zeroing, no read-modify-write and no barrier between
// children. `per` workgroups per front, each `cols` columns (by rch ranges of rlen rows where one
// child's inverse map would not fit); a wavefront takes four columns by 64 rows at a time, whose
// children follow from one ballot, three children's entries (kAsmAhead, twelve loads) in flight.
// Bound by round trips (record, children, maps, entries): 7 us for a few fronts of 100 rows and 29 us a
// height on average on the 164k icosphere, where scattering into the front in memory, child by child,
// took 13 and 41.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
constexpr int kAsmAhead = 3;   // children whose entries are loaded together (four columns each)
constexpr int kAsmBatch = 64;  // children whose maps are inverted at a time (one per lane)
__global__ __launch_bounds__(kFacBlock) void k_fac_assemble(FacArgs A, int h0, FacAssembly as) {
    const FacDev S = A.sn[h0 + blockIdx.x / as.per];
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, w = S.w, no = S.noff, m = S.m;
    if (A.stamp && h0 == 0 && blockIdx.x == 0 && tid == 0) *A.stamp = wall_clock64();
    const int part = (int)(blockIdx.x % as.per), t0 = part / as.rch * as.cols, t1 = min(m, t0 + as.cols);
    const int r0 = max(t0, part % as.rch * as.rlen), r1 = min(m, (part % as.rch + 1) * as.rlen), len = r1 - r0;
    if (t0 >= m || len <= 0) return;
    MD_G double *P = A.P + S.poff, *U = A.U + S.uoff;
    const MD_G int *rows = A.offrows + S.roff;
    extern __shared__ int inv[];        // row r of child c of the batch at c * len + r - r0
    __shared__ double obuf[4][4][64];   // original entries of a wavefront's quad
    int *rsh = inv + as.ninv;           // the front's row list, for the searches of the original entries
    const bool staged = t0 < w && no <= as.nrows;
    if (staged)
        for (int e = tid; e < no; e += kFacBlock) rsh[e] = rows[e];
    // waves over column quads first, then over their row chunks
    const int nq = (t1 - t0 + 3) / 4, wq = min(4, nq >= 3 ? 4 : nq), wc = 4 / wq;
    const int nch = S.ce - S.cb, cap = min(kAsmBatch, as.ninv / len);
    int cb = 0;
    do {
        const int nb = min(nch - cb, cap);
        FacChild C{0, 0, 0};
        if (lane < nb) C = A.child[S.cb + cb + lane];
        if (cb > 0) __syncthreads();  // the previous batch's maps are read
        for (int e = tid; e < nb * len; e += kFacBlock) inv[e] = -1;
        __syncthreads();
        for (int c = wv; c < nb; c += 4) {
            const int nc = __builtin_amdgcn_readlane(C.noff, c), roff = __builtin_amdgcn_readlane(C.roff, c);
            for (int a = lane; a < nc; a += 64) {
                const int r = A.rel[roff + a];
                if (r >= r0 && r < r1) inv[c * len + r - r0] = a;
                if (r >= m) *A.flag = 2;
            }
        }
        __syncthreads();
        for (int q = wv % wq; q < nq; q += wq) {
            const int tq = t0 + 4 * q;
            // rows of the quad's columns in the children (lane: child), -1: none
            int cbm[4];
            unsigned long long any = 0;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int t = tq + g;
                cbm[g] = -1;
                if (lane < nb && t < t1) {
                    if (t >= r0 && t < r1) {
                        cbm[g] = inv[lane * len + t - r0];
                    } else {  // above a later row range
                        int lo = 0, hi = C.noff;
                        while (lo < hi) {
                            const int mid = (lo + hi) >> 1;
                            if (A.rel[C.roff + mid] < t) lo = mid + 1;
                            else hi = mid;
                        }
                        if (lo < C.noff && A.rel[C.roff + lo] == t) cbm[g] = lo;
                    }
                }
                any |= __ballot(cbm[g] >= 0);
            }
            // original entries of pivot columns: lane 16 g + i holds slot i of column tq + g (and of
            // i + 16, ... below): its front row, or -1
            const int og = lane >> 4, ot = tq + og, oi = lane & 15;
            const bool opiv = cb == 0 && ot < min(w, t1);
            const int oj = S.c0 + ot, osl = opiv ? oj / kSlice : 0, ol = oj % kSlice;
            const int oq0 = opiv ? A.slice_ptr[osl] : 0, oq1 = opiv ? A.slice_ptr[osl + 1] : 0;
            auto original = [&](int x, int &row, double &val) {
                row = -1;
                val = 0.0;
                if (oq0 + x >= oq1) return;
                const long long gs = (long long)(oq0 + x) * kSlice + ol;
                const int i = A.sell_col[gs];
                if (i <= oj || i >= A.nf) return;
                val = -A.w64[gs];
                row = i - S.c0;
                if (row < w) return;
                int lo = 0, hi = no;  // first off row >= i
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if ((staged ? rsh[mid] : rows[mid]) < i) lo = mid + 1;
                    else hi = mid;
                }
                if (lo < no && (staged ? rsh[lo] : rows[lo]) == i) row = w + lo;
                else { row = -1; *A.flag = 2; }
            };
            int orow;
            double oval;
            original(oi, orow, oval);
            const double odiag = opiv && oi == 0 ? A.diag[oj] : 0.0;
            for (int ch = wv / wq; tq + 64 * ch < r1; ch += wc) {
                double acc[4];
                int r[4];
                bool on[4];
                MD_G double *dst[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int t = tq + g;
                    r[g] = t + 64 * ch + lane;
                    on[g] = t < t1 && r[g] >= r0 && r[g] < r1;
                    dst[g] = t >= w ? U + (long long)(t - w) * no + (r[g] - w) : P + (long long)t * m + r[g];
                    acc[g] = cb > 0 && on[g] ? *dst[g] : 0.0;
                }
                if (cb == 0 && tq < w) {
                    // through LDS: clear the quad's 4 x 64 entries, put the original ones, take them
                    // (one wavefront: its LDS accesses are in order)
                    double (*ob)[64] = obuf[wv];
#pragma unroll
                    for (int g = 0; g < 4; ++g) ob[g][lane] = 0.0;
                    wave_lds_fence();
                    const int lo = ot + 64 * ch;
                    if (opiv && oi == 0 && ch == 0) ob[og][0] = odiag;
                    if (orow >= lo && orow < lo + 64) ob[og][orow - lo] = oval;
                    for (int x = oi + 16; __any(oq0 + x < oq1); x += 16) {
                        int row;
                        double val;
                        original(x, row, val);
                        if (row >= lo && row < lo + 64) ob[og][row - lo] = val;
                    }
                    wave_lds_fence();
#pragma unroll
                    for (int g = 0; g < 4; ++g) acc[g] = ob[g][lane];
                    wave_lds_fence();
                }
                for (unsigned long long todo = any; todo;) {
                    double v[kAsmAhead][4];
#pragma unroll
                    for (int k = 0; k < kAsmAhead; ++k) {
                        const bool has = todo != 0;
                        const int c = has ? __builtin_ctzll(todo) : 0;
                        todo &= todo - 1;
                        const int nc = __builtin_amdgcn_readlane(C.noff, c);
                        const unsigned long long uo =
                            (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)C.uoff, c) |
                            (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(C.uoff >> 32), c) << 32;
                        const MD_G double *Uc = A.U + (long long)uo;
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const int bcol = __builtin_amdgcn_readlane(cbm[g], c);
                            const int a = has && bcol >= 0 && on[g] ? inv[c * len + r[g] - r0] : -1;
                            v[k][g] = a >= 0 ? Uc[(long long)bcol * nc + a] : 0.0;
                        }
                    }
#pragma unroll
                    for (int k = 0; k < kAsmAhead; ++k)
#pragma unroll
                        for (int g = 0; g < 4; ++g) acc[g] += v[k][g];
                }
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    if (on[g]) *dst[g] = acc[g];
            }
        }
        cb += nb;
    } while (cb < nch);
}

// Fronts are factored by symmetric block sweeps. A sweep on the columns of block s with S = A_ss^{-1}
// maps A_ss -> -S, A_Is -> A_Is S, A_IJ -> A_IJ - A_Is S A_Js^T; it keeps the matrix symmetric, and
// after the sweeps on a front's pivot blocks it holds [-D^{-1}, G^T; G, U]: the sweeps' panels and the
// update matrix for the parent. Swept at 64 columns over the front (k_fac_inv0, k_fac_step), at 16
// within a 64 x 64 block (invert64), at 4 within a 16 x 16 block (sweep_panel); k_fac_small sweeps a
// whole small front by panels of 4 pivots.
// LDS rows of the 64 x 64 operands, in doubles (odd: a column of a row-major tile hits 32 banks)
constexpr int kLdT = kFb + 1;

// v_mfma_f64_16x16x4f64: A(i, k) from lane i + 16 k, B(k, j) from lane j + 16 k, D(i, j) in lane
// j + 16 (i % 4), register i / 4. Register c of a D block is the B operand of k in [4 c, 4 c + 4), and
// for a symmetric block also its transpose's A operand.
typedef double dv4 __attribute__((ext_vector_type(4)));
#define MD_MFMA64(a, b, c) __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0)

__device__ __forceinline__ double f64_of(unsigned lo, unsigned hi) {
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// x[t] = p of lane (lane % 16) + 16 t, in every lane: the four rows of 16 lanes to all rows
// (v_permlane16_swap exchanges odd rows of one operand with even rows of the other, v_permlane32_swap
// the halves).
__device__ __forceinline__ void rows4(double p, double (&x)[4]) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, p);
    const unsigned w[2] = {(unsigned)u, (unsigned)(u >> 32)};
    unsigned r[4][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const auto a = __builtin_amdgcn_permlane16_swap(w[h], w[h], false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false);
        const auto c = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);
        r[0][h] = b[0]; r[2][h] = b[1]; r[1][h] = c[0]; r[3][h] = c[1];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = f64_of(r[t][0], r[t][1]);
}

// v of lane N of each row of 16 lanes, to the whole row (DPP row_newbcast).
template <int N>
__device__ __forceinline__ double row_bcast(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)u, 0x150 + N, 0xF, 0xF, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)(unsigned)(u >> 32), 0x150 + N, 0xF, 0xF, true);
    return f64_of(lo, hi);
}

// 1 / d: v_rcp_f64 (relative error below 2^-22) and y (1 + e + e^2), e = 1 - d y.
__device__ __forceinline__ double recip64(double d) {
    double y = __builtin_amdgcn_rcp(d);
    const double e = __builtin_fma(-d, y, 1.0);
    return __builtin_fma(y, __builtin_fma(e, e, e), y);
}

// Sweep of a symmetric matrix of NB x NB blocks of 16 x 16 (all blocks stored, in the layout of D),
// by one wavefront, on the four columns 4 C .. 4 C + 3 of block 0 (PARTIAL: on the first cnt of
// them). Register C of block (0, J) holds a(16 J + j, 4 C + k) at lane j + 16 k: the panel is one
// register per block, already in the layout of both operands of the rank-4 update, one MFMA per
// block. W = P B^{-1} (B the panel's 4 x 4 pivot block) comes from B's LDL^T, whose entries every lane
// forms for itself, and a substitution along the lane's row; the rows of the panel itself are solved
// for minus the unit rows, which gives -B^{-1}. The columns of the panel are cleared and their B
// operand set to minus the unit columns, so that the update leaves W there, exactly.
// Pivots with index < real must exceed thr, else bad is set.
template <int NB, int C, bool PARTIAL>
__device__ __forceinline__ void sweep_panel(dv4 (&a)[NB][NB], int lane, int cnt, int real, double thr, bool &bad) {
    const int j = lane & 15, g = lane >> 4, jj = j & 3;
    double x[4];
    rows4(a[0][0][C], x);
    const double d0 = row_bcast<4 * C>(x[0]);
    double a10 = row_bcast<4 * C + 1>(x[0]), a20 = row_bcast<4 * C + 2>(x[0]), a30 = row_bcast<4 * C + 3>(x[0]);
    double a11 = row_bcast<4 * C + 1>(x[1]), a21 = row_bcast<4 * C + 2>(x[1]), a31 = row_bcast<4 * C + 3>(x[1]);
    double a22 = row_bcast<4 * C + 2>(x[2]), a32 = row_bcast<4 * C + 3>(x[2]), a33 = row_bcast<4 * C + 3>(x[3]);
    if (PARTIAL) {  // pivots past cnt: the unit matrix
        if (cnt < 2) { a10 = 0.0; a21 = 0.0; a31 = 0.0; a11 = 1.0; }
        if (cnt < 3) { a20 = 0.0; a21 = 0.0; a32 = 0.0; a22 = 1.0; }
        if (cnt < 4) { a30 = 0.0; a31 = 0.0; a32 = 0.0; a33 = 1.0; }
    }
    const double r0 = recip64(d0);
    const double l10 = a10 * r0, l20 = a20 * r0, l30 = a30 * r0;
    const double d1 = __builtin_fma(-l10, a10, a11), r1 = recip64(d1);
    const double b21 = __builtin_fma(-l10, a20, a21), b31 = __builtin_fma(-l10, a30, a31);
    const double b22 = __builtin_fma(-l20, a20, a22), b32 = __builtin_fma(-l20, a30, a32), b33 = __builtin_fma(-l30, a30, a33);
    const double l21 = b21 * r1, l31 = b31 * r1;
    const double d2 = __builtin_fma(-l21, b21, b22), r2 = recip64(d2);
    const double c32 = __builtin_fma(-l21, b31, b32), c33 = __builtin_fma(-l31, b31, b33);
    const double l32 = c32 * r2;
    const double d3 = __builtin_fma(-l32, c32, c33), r3 = recip64(d3);
    if ((4 * C < real && !(d0 > thr)) || (4 * C + 1 < real && !(d1 > thr)) || (4 * C + 2 < real && !(d2 > thr)) ||
        (4 * C + 3 < real && !(d3 > thr)))
        bad = true;
    double w[NB], p[NB];
#pragma unroll
    for (int J = 0; J < NB; ++J) {
        const bool inp = J == 0 && (j >> 2) == C && (!PARTIAL || jj < cnt);
        const double P = a[0][J][C];
        if (J > 0) rows4(P, x);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (PARTIAL && t >= cnt) x[t] = 0.0;
            if (J == 0) x[t] = inp ? (jj == t ? -1.0 : 0.0) : x[t];
        }
        const double u1 = __builtin_fma(-l10, x[0], x[1]);
        const double u2 = __builtin_fma(-l21, u1, __builtin_fma(-l20, x[0], x[2]));
        const double u3 = __builtin_fma(-l32, u2, __builtin_fma(-l31, u1, __builtin_fma(-l30, x[0], x[3])));
        const double w3 = u3 * r3;
        const double w2 = __builtin_fma(-l32, w3, u2 * r2);
        const double w1 = __builtin_fma(-l31, w3, __builtin_fma(-l21, w2, u1 * r1));
        const double w0 = __builtin_fma(-l30, w3, __builtin_fma(-l20, w2, __builtin_fma(-l10, w1, x[0] * r0)));
        w[J] = g == 0 ? w0 : g == 1 ? w1 : g == 2 ? w2 : w3;
        p[J] = inp ? (g == jj ? -1.0 : 0.0) : P;
        if (J == 0) {
#pragma unroll
            for (int I = 0; I < NB; ++I)
#pragma unroll
                for (int k = 0; k < 4; ++k) a[I][0][k] = inp ? 0.0 : a[I][0][k];
        }
    }
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int J = 0; J < NB; ++J) a[I][J] = MD_MFMA64(-w[I], p[J], a[I][J]);
#pragma unroll
    for (int J = 0; J < NB; ++J) a[0][J][C] = !PARTIAL || g < cnt ? w[J] : a[0][J][C];
}

// LDS of invert64: the inverse of the current 16 x 16 diagonal block and the current block column,
// two buffers each.
constexpr int kIb = 16, kIbLd = kIb + 1;
struct InvLds {
    double s[2][kIb][kIbLd];
    double a[2][4][kIb][kIbLd];
};
static_assert(kFb == 4 * kIb, "one block column of 16 per wavefront");

static_assert(kFacBlock == 4 * 64, "four wavefronts");

// The symmetric 64 x 64 block in m (lower part, row r at r * kLdT) replaced by minus its inverse
// in the layout of D: wave v holds block column v in acc. b < 64: the leading b x b block (rows and
// columns past it are taken as the identity, and 16-blocks past it are not swept). Ends without a
// barrier; work may not alias m. Step K: wave K sweeps its diagonal block and publishes its inverse
// and the block column; after one barrier the other waves form T_J = S A_KJ and update their columns,
// A_IJ -= A_IK T_J, and wave K forms A_IK S. A loop over K: the block rows rotate (row K is acc[0]), for
// nothing, since an MFMA may write another register than it adds to; unrolled, the code of this and its
// callers outgrew the instruction cache, and its fetch was a third of a launch.
// A chain of b pivots: per 16 of them 2,950 cycles of dependent FP64 arithmetic in the panel sweeps
// (DPP and permlane broadcasts in place of LDS) and 1,900 for the exchange and the updates (one
// v_mfma_f64_16x16x4 per 16 cycles and CU): 19,400 for 64. As k_fac_inv0 runs it, its code not yet in the
// instruction cache, 24,000 (10 us of the kernel's 15; loading the block takes 4, storing the inverse 0.7).
__device__ __forceinline__ void invert64(const double *m, InvLds &work, int b, double thr, dv4 (&acc)[4], bool &bad) {
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int r = kIb * I + 4 * c + g, q = kIb * wv + j;
            acc[I][c] = r < b && q < b ? m[max(r, q) * kLdT + min(r, q)] : r == q ? 1.0 : 0.0;
        }
    const int nk = (b + kIb - 1) / kIb;
#pragma unroll 1
    for (int K = 0; K < 4; ++K) {
        dv4 out[4];
        if (K < nk) {
            double (*Ss)[kIbLd] = work.s[K & 1];
            double (*Sa)[kIb][kIbLd] = work.a[K & 1];
            if (wv == K) {
#pragma unroll
                for (int I = 1; I < 4; ++I)
#pragma unroll
                    for (int c = 0; c < 4; ++c) Sa[I][4 * c + g][j] = acc[I][c];
                dv4 d[1][1];
                d[0][0] = acc[0];
                const int real = b - kIb * K;
                sweep_panel<1, 0, false>(d, lane, 4, real, thr, bad);
                sweep_panel<1, 1, false>(d, lane, 4, real, thr, bad);
                sweep_panel<1, 2, false>(d, lane, 4, real, thr, bad);
                sweep_panel<1, 3, false>(d, lane, 4, real, thr, bad);
                out[3] = d[0][0];
#pragma unroll
                for (int c = 0; c < 4; ++c) Ss[4 * c + g][j] = -out[3][c];
            }
            __syncthreads();
            if (wv == K) {
#pragma unroll
                for (int I = 1; I < 4; ++I) out[I - 1] = dv4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int I = 1; I < 4; ++I) out[I - 1] = MD_MFMA64(Sa[I][j][4 * c + g], -out[3][c], out[I - 1]);
            } else {
                dv4 t = dv4{0.0, 0.0, 0.0, 0.0}, t2 = t;
#pragma unroll
                for (int c = 0; c < 4; c += 2) {
                    t = MD_MFMA64(Ss[j][4 * c + g], acc[0][c], t);
                    t2 = MD_MFMA64(Ss[j][4 * c + 4 + g], acc[0][c + 1], t2);
                }
                t += t2;
#pragma unroll
                for (int I = 1; I < 4; ++I) out[I - 1] = acc[I];
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int I = 1; I < 4; ++I) out[I - 1] = MD_MFMA64(-Sa[I][j][4 * c + g], t[c], out[I - 1]);
                out[3] = t;
            }
        } else {  // rotate only
#pragma unroll
            for (int I = 0; I < 4; ++I) out[I] = acc[(I + 1) & 3];
        }
#pragma unroll
        for (int I = 0; I < 4; ++I) acc[I] = out[I];
    }
}

// Block s of a front, complete in m (LDS): S = A_ss^{-1} into block (s, s) of the workspace `out`.
__device__ __forceinline__ void pivot_inverse(const FacArgs &A, const FacDev &S, int s, const double *m, InvLds &work,
                                              const FrontBuf &out) {
    const int kb = s * kFb, b = min(kFb, S.w - kb);
    const double thr = pivot_floor(A);
    dv4 acc[4];
    bool bad = false;
    invert64(m, work, b, thr, acc, bad);
    if (bad && (threadIdx.x & 63) == 0) *A.flag = 1;
    const int wv = threadIdx.x >> 6, j = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4, r = kIb * wv + j;
    if (r >= b) return;
    MD_G double *p = out.d + (long long)(kb + g) * out.ldd + kb + r;  // entry (r, q) = (q, r): lanes along r
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int q = kIb * I + 4 * c;
            if (q + g < b) p[q * out.ldd] = -acc[I][c];
        }
}

// Block 0 of the fronts of a height (one workgroup per front).
__global__ __launch_bounds__(kFacBlock) void k_fac_inv0(FacArgs A, int h0) {
    const FacDev S = A.sn[h0 + blockIdx.x];
    __shared__ double m[kFb * kLdT];
    __shared__ InvLds work;
    const FrontBuf B = front_buf(A, S, 0);
    const int b = min(kFb, S.w), r = threadIdx.x % kFb;
#pragma unroll
    for (int i = 0; i < kFb * kFb / kFacBlock; ++i) {
        const int c = threadIdx.x / kFb + 4 * i;
        if (r < b && c <= r) m[r * kLdT + c] = B.d[c * B.ldd + r];
    }
    __syncthreads();
    pivot_inverse(A, S, 0, m, work, B);
}

// ---- FP64 products of the sweeps on the matrix cores ---------------------------------------
//
// A 64 x 64 output tile per workgroup of 256 threads: wave v computes rows [32 (v / 2), +32) and
// columns [32 (v % 2), +32) as 2 x 2 blocks of v_mfma_f64_16x16x4, with both operands whole in LDS
// (64 values of k, rows kLdT apart).

struct MmaAcc {
    dv4 c[2][2];
};

__device__ __forceinline__ void mma_zero(MmaAcc &acc) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc.c[x][y] = dv4{0.0, 0.0, 0.0, 0.0};
}

// Tile coordinates (i, j) within the 64 x 64 output of this thread's element (x, y, r).
__device__ __forceinline__ int mma_row(int x, int r) {
    return 32 * ((threadIdx.x / 64) >> 1) + 16 * x + 4 * r + ((threadIdx.x & 63) >> 4);
}
__device__ __forceinline__ int mma_col(int y) { return 32 * ((threadIdx.x / 64) & 1) + 16 * y + (threadIdx.x & 15); }

// acc(i, j) += sum_{k < kn} Ar[k][i] Bc[k][j], 16 values of k per turn (operands past kn are zero).
__device__ __forceinline__ void mma_span(const double *Ar, const double *Bc, int kn, MmaAcc &acc) {
    const int wv = threadIdx.x / 64, lane = threadIdx.x & 63;
    const double *ap = Ar + (lane >> 4) * kLdT + 32 * (wv >> 1) + (lane & 15);
    const double *bp = Bc + (lane >> 4) * kLdT + 32 * (wv & 1) + (lane & 15);
    for (int k = 0; k < kn; k += 16, ap += 16 * kLdT, bp += 16 * kLdT) {
        double a[4][2], b[4][2];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                a[u][y] = ap[4 * u * kLdT + 16 * y];
                b[u][y] = bp[4 * u * kLdT + 16 * y];
            }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) acc.c[x][y] = MD_MFMA64(a[u][x], b[u][y], acc.c[x][y]);
    }
}

// fn(value, row, column) over this thread's accumulators.
template <class Fn>
__device__ __forceinline__ void mma_each(const MmaAcc &acc, Fn fn) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) fn(acc.c[x][y][r], mma_row(x, r), mma_col(y));
}

// Lower block (I, J), I >= J, of the q-th tile of a lower-triangular tile grid.
__device__ __forceinline__ void lower_tile(int q, int &I, int &J) {
    int i = 0;
    while ((i + 1) * (i + 2) / 2 <= q) ++i;
    I = i;
    J = q - i * (i + 1) / 2;
}

constexpr int kTileVals = kFb * kFb / kFacBlock;  // values of a 64 x 64 tile per thread
static_assert(kFacBlock == 4 * kFb, "four columns of a tile per pass of the workgroup");

// Block (X, s) of a front (X: pivot blocks 0 .. nb - 1, then blocks of 64 off rows) from its lower
// tiles, into registers and from there to LDS as Z[t][x] = A(x of block X, t of block s): from block s
// down the tile itself, above it the transpose of tile (s, X). Zero past the matrix.
__device__ __forceinline__ void block_fetch(const FrontBuf &B, int w, int no, int nb, int X, int s, double (&v)[kTileVals]) {
    const int lo = threadIdx.x % kFb, hi = threadIdx.x / kFb;
    const int col = (X >= s ? s : X) * kFb + hi;
    const bool off = X >= nb;
    const int row = off ? (X - nb) * kFb + lo : (X >= s ? X : s) * kFb + lo;
    const long long ld = off ? B.ldf : B.ldd;
    const MD_G double *p = (off ? B.f : B.d) + col * ld + row;
    const bool in = row < (off ? no : w);
#pragma unroll
    for (int i = 0; i < kTileVals; ++i) v[i] = in && col + 4 * i < w ? p[4 * i * ld] : 0.0;
}
__device__ __forceinline__ void block_put(bool below, const double (&v)[kTileVals], double *Z) {
    const int lo = threadIdx.x % kFb, hi = threadIdx.x / kFb, z = below ? hi * kLdT + lo : lo * kLdT + hi;
    const int step = below ? 4 * kLdT : 4;
#pragma unroll
    for (int i = 0; i < kTileVals; ++i) Z[z + i * step] = v[i];
}

// Step s of the block sweeps over the fronts of a height (`per` lower tiles of 64 x 64 per front, its
// off rows and update matrix included): tile (I, J) from S = A_ss^{-1}, in one launch: with W = A_Is S
// (64 x 64, in LDS), A_IJ - W A_Js^T; W itself in block column s; -S on the diagonal. The workgroup of
// tile (s + 1, s + 1), scheduled first, inverts it for the next step while the other tiles still run.
// The last step of a front writes its panels: D^{-1} (minus the swept pivot block) and G. Tiles leave
// through LDS, so one short loop stores every kind.
// Bound by the chain of one tile per step: load, two products (1.7 us each at one MFMA per 16 cycles
// and CU) and the inversion (8 to 10): 20 us a step of the 164k icosphere's top heights, whose other tiles
// run on CUs that the chain leaves idle. So the off rows and the update matrix are swept along: as
// products after the sweeps (G = F D^{-1}, U -= G F^T, split over K) they took another 20 to 105 us a
// height, waiting on their own chunks.
__global__ __launch_bounds__(kFacBlock) __attribute__((amdgpu_waves_per_eu(2))) void k_fac_step(FacArgs A, int h0, int s, int per) {
    const FacDev S = A.sn[h0 + blockIdx.x / per];
    const int w = S.w, no = S.noff, nb = (w + kFb - 1) / kFb, nbo = nb + (no + kFb - 1) / kFb;
    if (s >= nb) return;
    int q = (int)(blockIdx.x % per);
    if (q >= nbo * (nbo + 1) / 2) return;
    const bool last = s == nb - 1;
    if (!last) {  // tile 0 and tile (s + 1, s + 1) trade places
        const int d = (s + 1) * (s + 2) / 2 + s + 1;
        q = q == 0 ? d : q == d ? 0 : q;
    }
    int I, J;
    lower_tile(q, I, J);
    const FrontBuf B = front_buf(A, S, s), O = front_buf(A, S, s + 1);
    __shared__ double Za[kFb * kLdT], Zb[kFb * kLdT];
    static_assert(sizeof(InvLds) <= sizeof(Za), "the inversion works in the first operand's place");
    const int X = I == s ? J : I;  // W = A_Xs S
    const bool inner = I != s && J != s, upd = J >= nb;
    const int kn = (min(kFb, w - s * kFb) + 3) & ~3;
    // where the tile's entries are: rows, columns, and those of the tile within bounds
    const int i0 = (I < nb ? I : I - nb) * kFb, j0 = (upd ? J - nb : J) * kFb;
    const int rn = min(kFb, (I < nb ? w : no) - i0), cn = min(kFb, (upd ? no : w) - j0);
    MD_G double *U = A.U + S.uoff;
    double vs[kTileVals], vx[kTileVals], vj[kTileVals];
    block_fetch(B, w, no, nb, s, s, vs);  // S, both triangles
    if (X != s) block_fetch(B, w, no, nb, X, s, vx);
    if (inner && I != J) block_fetch(B, w, no, nb, J, s, vj);
    double own[2][2][4];  // the tile's own entries, where the accumulators will be (row c, column r)
    if (inner) {
        const int c0 = mma_row(0, 0), r0 = mma_col(0);
        const long long ld = upd ? no : I < nb ? B.ldd : B.ldf;
        const MD_G double *p = (upd ? U : I < nb ? B.d : B.f) + (j0 + c0) * ld + i0 + r0;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    own[x][y][r] = r0 + 16 * y < rn && c0 + 16 * x + 4 * r < cn ? p[(16 * x + 4 * r) * ld + 16 * y] : 0.0;
    }
    block_put(true, vs, Za);
    if (X != s) {
        block_put(X > s, vx, Zb);
        __syncthreads();
        MmaAcc acc;
        mma_zero(acc);
        mma_span(Za, Zb, kn, acc);  // (k, r): W(r, k)
        __syncthreads();
        mma_each(acc, [&](double v, int k, int r) { Za[k * kLdT + r] = v; });
        if (inner) {
            if (I != J) block_put(J > s, vj, Zb);
            __syncthreads();
            mma_zero(acc);
            mma_span(Zb, Za, kn, acc);  // (c, r): sum_k A_Js(c, k) W(r, k)
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc.c[x][y][r] = own[x][y][r] - acc.c[x][y][r];
            __syncthreads();  // the operands are read
            if (!last && I == s + 1 && J == s + 1) {
                mma_each(acc, [&](double v, int c, int r) { if (r >= c) Zb[r * kLdT + c] = v; });
                __syncthreads();
                pivot_inverse(A, S, s + 1, Zb, *reinterpret_cast<InvLds *>(Za), O);
                return;
            }
            mma_each(acc, [&](double v, int c, int r) { Za[c * kLdT + r] = v; });
        }
    }
    __syncthreads();
    // Za: entry (r, c) of the tile at c * kLdT + r (S itself on the diagonal, negated below), except that
    // in block row s it holds W_J(r', k) for entry (k, r')
    const bool swap = I == s && J != s, dinv = last && I < nb;
    const double sign = (X == s) != dinv ? -1.0 : 1.0;  // -S on the diagonal; D^{-1} is minus the swept block
    auto entry = [&](int r, int c) { return sign * Za[swap ? r * kLdT + c : c * kLdT + r]; };
    const int lo = threadIdx.x % kFb, hi = threadIdx.x / kFb;
    if (!last || upd) {
        const long long ld = upd ? no : I < nb ? O.ldd : O.ldf;
        MD_G double *p = (upd ? U : I < nb ? O.d : O.f) + j0 * ld + i0;
        if (lo < rn)
            for (int c = hi; c < cn; c += 4) p[c * ld + lo] = entry(lo, c);
        return;
    }
    auto put = [&](MD_G void *dst, long long o, double v) {
        if (A.solve64) static_cast<MD_G double *>(dst)[o] = v;
        else static_cast<MD_G float *>(dst)[o] = (float)v;
    };
    // row-major panel [D^{-1}; G], lanes along its columns; the pivot rows' tiles also mirrored (the
    // diagonal tile from its lower part), G also to the column-major panel
    const long long pr = S.pr_off + (long long)((dinv ? 0 : w) + i0) * w + j0;
    if (lo < cn)
        for (int r = hi; r < rn; r += 4) put(A.pr, pr + (long long)r * w + lo, I == J ? entry(max(r, lo), min(r, lo)) : entry(r, lo));
    if (I == J || lo >= rn) return;
    for (int c = hi; c < cn; c += 4) {
        if (dinv) put(A.pr, S.pr_off + (long long)(j0 + c) * w + i0 + lo, entry(lo, c));
        else put(A.pc, S.pc_off + (long long)(j0 + c) * no + i0 + lo, entry(lo, c));
    }
}

// The front in LDS (symmetric, row r at r * LD, zero past its m rows) of m <= 16 NB rows, swept on its w
// pivots by one wavefront with all of it in registers, and put back: [-D^{-1}, G^T; G, U]. After the
// sweeps of block 0's columns the blocks rotate (block k to k - 1), so every panel has fixed
// registers.
template <int NB, int LD>
__device__ __forceinline__ bool small_front(double *Fs, int w, double thr) {
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    dv4 a[NB][NB];
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int J = 0; J < NB; ++J)
#pragma unroll
            for (int c = 0; c < 4; ++c) a[I][J][c] = Fs[(kIb * I + 4 * c + g) * LD + kIb * J + j];
    bool bad = false;
    int rot = 0;
#pragma unroll 1
    for (int k0 = 0; k0 < w; k0 += kIb) {
        const int left = w - k0;
        sweep_panel<NB, 0, true>(a, lane, min(4, left), left, thr, bad);
        if (left > 4) sweep_panel<NB, 1, true>(a, lane, min(4, left - 4), left, thr, bad);
        if (left > 8) sweep_panel<NB, 2, true>(a, lane, min(4, left - 8), left, thr, bad);
        if (left > 12) sweep_panel<NB, 3, true>(a, lane, min(4, left - 12), left, thr, bad);
        dv4 t[NB][NB];
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
            for (int J = 0; J < NB; ++J) t[I][J] = a[(I + 1) % NB][(J + 1) % NB];
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
            for (int J = 0; J < NB; ++J) a[I][J] = t[I][J];
        rot = rot + 1 == NB ? 0 : rot + 1;
    }
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int J = 0; J < NB; ++J) {
            const int bi = I + rot >= NB ? I + rot - NB : I + rot, bj = J + rot >= NB ? J + rot - NB : J + rot;
            double *dst = Fs + (kIb * bi + g) * LD + kIb * bj + j;
#pragma unroll
            for (int c = 0; c < 4; ++c) dst[4 * c * LD] = a[I][J][c];
        }
    return bad;
}

// Small fronts (m = w + noff <= 16 NB), one workgroup per front: assembly in LDS (the original
// entries, then the children's update matrices in child order, as k_fac_assemble adds them; the
// front's row list staged in LDS for the searches) by all of its BLOCK threads, the sweeps by its
// first wavefront in registers (small_front), and all of it out again: D^{-1} and G to the sweeps'
// panels, U for the parent. BLOCK is 64 for many fronts (the leaves, which have no children) and 256
// for few, where the additions of the children are the longer part; fronts of more than 48 rows, which
// have children and whose LDS and registers hold four wavefronts' fronts per CU, take 128 where they
// are many. Limited to two wavefronts per SIMD's registers (256), which 260 had halved. The FP64
// panel workspace is not used. 50 us for the 6,616 leaves of the 164k icosphere, 70 for its 2,449 fronts of up to
// 64 rows above them (92 with one wavefront each) and 14 us for a single front of 52 columns; the
// column-by-column Cholesky in LDS that stood here took 100 us for the leaves and 88 for the single one.
constexpr int kSmallSlotLanes = 4;  // lanes per pivot column for its original entries
constexpr int kSmallAhead = 16;     // columns of a child's update matrix in flight
template <int BLOCK, int NB>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2))) void k_fac_small(FacArgs A, int h0) {
    const FacDev S = A.sn[h0 + blockIdx.x];
    const int tid = threadIdx.x, w = S.w, no = S.noff, m = S.m;
    if (A.stamp && h0 == 0 && blockIdx.x == 0 && tid == 0) *A.stamp = wall_clock64();
    if (m > kIb * NB) {  // the host sends only small fronts
        if (tid == 0) *A.flag = 2;
        return;
    }
    constexpr int LD = kIb * NB + 1;
    __shared__ double Fs[kIb * NB * LD];
    __shared__ int rows[kIb * NB];
    for (int e = tid; e < no; e += BLOCK) rows[e] = A.offrows[S.roff + e];
    const bool narrow = NB > 2 && m <= 2 * kIb;  // swept as two blocks
    for (int e = tid; e < (narrow ? 2 * kIb : NB * kIb) * LD; e += BLOCK) Fs[e] = 0.0;
    __syncthreads();
    // original entries, kSmallSlotLanes lanes per pivot column (one slot each; every front entry
    // receives at most one)
    for (int k = tid / kSmallSlotLanes; k < w; k += BLOCK / kSmallSlotLanes) {
        const int j = S.c0 + k, sl = j / kSlice, l = j % kSlice;
        if (tid % kSmallSlotLanes == 0) Fs[k * LD + k] = A.diag[j];
        for (int q = A.slice_ptr[sl] + tid % kSmallSlotLanes; q < A.slice_ptr[sl + 1]; q += kSmallSlotLanes) {
            const long long g = (long long)q * kSlice + l;
            const int i = A.sell_col[g];
            if (i <= j || i >= A.nf) continue;
            int r = i - S.c0;
            if (r >= w) {
                int lo = 0, hi = no;  // first off row >= i
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (rows[mid] < i) lo = mid + 1;
                    else hi = mid;
                }
                if (lo >= no || rows[lo] != i) {
                    *A.flag = 2;
                    continue;
                }
                r = w + lo;
            }
            Fs[r * LD + k] = -A.w64[g];
        }
    }
    __syncthreads();
    // children's update matrices in child order (distinct entries of one child land on distinct
    // front entries): a child has at most 64 rows, so its map is one register (the next child's in
    // flight), and kSmallAhead of its columns are loaded at a time
    const int wv = tid >> 6, lane = tid & 63;
    for (int cb = S.cb; cb < S.ce; cb += 64) {
        const int nb = min(S.ce - cb, 64);
        FacChild C{0, 0, 0};
        if (lane < nb) C = A.child[cb + lane];
        auto map_of = [&](int c) {
            const int nc = __builtin_amdgcn_readlane(C.noff, c), roff = __builtin_amdgcn_readlane(C.roff, c);
            return lane < nc ? A.rel[roff + lane] : -1;
        };
        int next = map_of(0);
        for (int c = 0; c < nb; ++c) {
            const int ra = next, nc = __builtin_amdgcn_readlane(C.noff, c);
            const unsigned long long uo = (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)C.uoff, c) |
                                          (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(C.uoff >> 32), c) << 32;
            const MD_G double *Uc = A.U + (long long)uo;
            if (c + 1 < nb) next = map_of(c + 1);
            if (nc > 64 || __any(ra >= m)) {  // the same in every wavefront
                *A.flag = 2;
                break;
            }
            for (int b0 = wv; b0 < nc; b0 += kSmallAhead * (BLOCK / 64)) {
                double v[kSmallAhead];
#pragma unroll
                for (int u = 0; u < kSmallAhead; ++u) {
                    const int col = b0 + u * (BLOCK / 64);
                    v[u] = col < nc && lane >= col && lane < nc ? Uc[(long long)col * nc + lane] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < kSmallAhead; ++u) {
                    const int col = b0 + u * (BLOCK / 64);
                    if (col >= nc) break;
                    const int rb = __builtin_amdgcn_readlane(ra, col);
                    if (lane >= col && lane < nc) Fs[ra * LD + rb] += v[u];
                }
            }
            __syncthreads();
        }
    }
    // the upper triangle from the lower one
    for (int e = tid; e < m * m; e += BLOCK) {
        const int r = e / m, c = e - r * m;
        if (c > r) Fs[r * LD + c] = Fs[c * LD + r];
    }
    __syncthreads();
    if (tid < 64) {
        const double thr = pivot_floor(A);
        bool bad;
        if (narrow) bad = small_front<2 < NB ? 2 : NB, LD>(Fs, w, thr);
        else bad = small_front<NB, LD>(Fs, w, thr);
        if (bad && tid == 0) *A.flag = 1;
    }
    __syncthreads();
    MD_G double *U = A.U + S.uoff;
    auto put = [&](MD_G void *dst, long long o, double v) {
        if (A.solve64) static_cast<MD_G double *>(dst)[o] = v;
        else static_cast<MD_G float *>(dst)[o] = (float)v;
    };
    // the sweeps' panels: row-major [D^{-1}; G] (m x w) and column-major G (no x w); U, lower part
    for (int e = tid; e < m * w; e += BLOCK) {
        const int r = e / w, c = e - r * w;
        const double v = Fs[r * LD + c];
        put(A.pr, S.pr_off + e, r < w ? -v : v);
    }
    for (int e = tid; e < no * w; e += BLOCK) {
        const int c = e / no, r = e - c * no;
        put(A.pc, S.pc_off + e, Fs[c * LD + w + r]);
    }
    for (int e = tid; e < no * no; e += BLOCK) {
        const int b = e / no, a = e - b * no;
        if (a >= b) U[e] = Fs[(w + b) * LD + w + a];
    }
}

// Plain device copy of n 16-byte elements (grid-stride): the known-size reference kernel for
// HBM counters and the achievable copy bandwidth.
__global__ __launch_bounds__(kBlock) void k_copy_probe(const f4 *__restrict__ src, f4 *__restrict__ dst, long long n) {
    const long long stride = (long long)gridDim.x * kBlock;
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

}  // namespace

template <int BLOCK>
static void fac_small_of(hipStream_t s, const FacArgs &A, int h0, int count, int mm) {
    const dim3 grid(count), block(BLOCK);
    if (mm <= kIb) hipLaunchKernelGGL((k_fac_small<BLOCK, 1>), grid, block, 0, s, A, h0);
    else if (mm <= 2 * kIb) hipLaunchKernelGGL((k_fac_small<BLOCK, 2>), grid, block, 0, s, A, h0);
    else hipLaunchKernelGGL((k_fac_small<BLOCK, 3>), grid, block, 0, s, A, h0);
}
void launch_fac_small(hipStream_t s, const FacArgs &A, int h0, int count, int mm) {
    if (count <= 0) return;
    if (mm > 3 * kIb) {
        if (count > kSmallManyWide) hipLaunchKernelGGL((k_fac_small<128, 4>), dim3(count), dim3(128), 0, s, A, h0);
        else hipLaunchKernelGGL((k_fac_small<256, 4>), dim3(count), dim3(256), 0, s, A, h0);
    } else if (count > kSmallManyFronts) {
        fac_small_of<64>(s, A, h0, count, mm);
    } else {
        fac_small_of<256>(s, A, h0, count, mm);
    }
}
void launch_fac_height(hipStream_t s, const FacArgs &A, int h0, int count, int nb, const FacAssembly &as, int tiles) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_fac_assemble, dim3(count * as.per), dim3(kFacBlock), sizeof(int) * (as.ninv + as.nrows), s, A, h0, as);
    hipLaunchKernelGGL(k_fac_inv0, dim3(count), dim3(kFacBlock), 0, s, A, h0);
    for (int b = 0; b < nb; ++b)
        hipLaunchKernelGGL(k_fac_step, dim3(count * tiles), dim3(kFacBlock), 0, s, A, h0, b, tiles);
}

void launch_copy_probe(hipStream_t s, const void *src, void *dst, long long n16) {
    if (n16 <= 0) return;
    hipLaunchKernelGGL(k_copy_probe, dim3(4096), dim3(kBlock), 0, s, static_cast<const f4 *>(src), static_cast<f4 *>(dst), n16);
}

#define MD_LAUNCH_T(kern, blocks, s, ...)                                                        \
    do {                                                                                        \
        if ((blocks) <= 0) return;                                                              \
        if (fp64) hipLaunchKernelGGL(kern<double>, dim3(blocks), dim3(kBlock), 0, s, __VA_ARGS__); \
        else hipLaunchKernelGGL(kern<float>, dim3(blocks), dim3(kBlock), 0, s, __VA_ARGS__);     \
    } while (0)

void launch_pcg_diag(hipStream_t s, LaunchSet L, int blocks, bool fp64) { MD_LAUNCH_T(k_pcg_diag, blocks, s, L); }
void launch_pcg_init(hipStream_t s, LaunchSet L, int blocks, bool fp64) { MD_LAUNCH_T(k_pcg_init, blocks, s, L); }
void launch_pcg_step(hipStream_t s, LaunchSet L, int blocks, int step, bool fp64) {
    MD_LAUNCH_T(k_pcg_step, blocks, s, L, step);
}
void launch_pcg_apply(hipStream_t s, LaunchSet L, int blocks, bool fp64) { MD_LAUNCH_T(k_pcg_apply, blocks, s, L); }

void launch_normals(hipStream_t s, LaunchSet Lf, int blocks_face, LaunchSet Ls, int blocks_slice, double *fn, d4 *out,
                    double *packed, const int *orig) {
    if (blocks_face > 0) hipLaunchKernelGGL(k_face_normals, dim3(blocks_face), dim3(kBlock), 0, s, Lf, fn);
    if (blocks_slice > 0)
        hipLaunchKernelGGL(k_vertex_normals, dim3(blocks_slice), dim3(kBlock), 0, s, Ls, (const double *)fn, out, packed, orig);
}

hipError_t scratch_address(void **ptr) {
    *ptr = nullptr;
    return hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch));
}

void launch_pack_xyz(hipStream_t s, const d4 *v, const int *internal, int n, double *dst, unsigned long long *stamp) {
    if (n > 0) hipLaunchKernelGGL(k_pack_xyz, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, v, internal, n, dst, stamp);
}
void launch_unpack_xyz(hipStream_t s, const UnpackArgs &a, bool fp64) {
    if (a.n <= 0) return;
    if (fp64) hipLaunchKernelGGL(k_unpack_xyz<double>, dim3((a.n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, a);
    else hipLaunchKernelGGL(k_unpack_xyz<float>, dim3((a.n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, a);
}
void launch_publish(hipStream_t s, unsigned long long *stamp, const int *flag, int *out) {
    if (stamp) hipLaunchKernelGGL(k_publish, dim3(1), dim3(1), 0, s, stamp, flag, out);
}

void launch_pack_results(hipStream_t s, const PackEntry *e, int count, int blocks) {
    if (count > 0 && blocks > 0) hipLaunchKernelGGL(k_pack_results, dim3(blocks), dim3(kBlock), 0, s, e, count);
}
void launch_scatter_entries(hipStream_t s, const TargetEntry *e, int k) {
    if (k > 0) hipLaunchKernelGGL(k_scatter_entries, dim3((k + kBlock - 1) / kBlock), dim3(kBlock), 0, s, e, k);
}

void launch_cotan_face(hipStream_t s, LaunchSet L, int blocks) {
    if (blocks > 0) hipLaunchKernelGGL(k_cotan_face, dim3(blocks), dim3(kBlock), 0, s, L);
}
void launch_cotan_slot(hipStream_t s, LaunchSet L, int blocks, double *diag, unsigned long long *amax) {
    if (blocks > 0) hipLaunchKernelGGL(k_cotan_slot, dim3(blocks), dim3(kBlock), 0, s, L, diag, amax);
}
void launch_local(hipStream_t s, LaunchSet L, int blocks, bool fp64) {
    if (blocks <= 0) return;
    if (fp64) hipLaunchKernelGGL(k_local<double>, dim3(blocks), dim3(kBlock), 0, s, L);
    else hipLaunchKernelGGL(k_local<float>, dim3(blocks), dim3(kBlock), 0, s, L);
}
void launch_residual(hipStream_t s, LaunchSet L, int blocks, bool fp64) {
    if (blocks <= 0) return;
    if (fp64) hipLaunchKernelGGL(k_residual<double>, dim3(blocks), dim3(kBlock), 0, s, L);
    else hipLaunchKernelGGL(k_residual<float>, dim3(blocks), dim3(kBlock), 0, s, L);
}
void launch_fwd(hipStream_t s, LaunchSet L, int blocks, int level, bool fp64) {
    if (blocks <= 0) return;
    if (blocks <= kPreloadMaxTiles) {
        if (fp64) hipLaunchKernelGGL((k_fwd<double, true>), dim3(blocks), dim3(kTile), 0, s, L, level);
        else hipLaunchKernelGGL((k_fwd<float, true>), dim3(blocks), dim3(kTile), 0, s, L, level);
    } else {
        if (fp64) hipLaunchKernelGGL((k_fwd<double, false>), dim3(blocks), dim3(kTile), 0, s, L, level);
        else hipLaunchKernelGGL((k_fwd<float, false>), dim3(blocks), dim3(kTile), 0, s, L, level);
    }
}
void launch_bwd(hipStream_t s, LaunchSet L, int blocks, int level, bool fp64) {
    if (blocks <= 0) return;
    if (blocks <= kPreloadMaxTiles) {
        if (fp64) hipLaunchKernelGGL((k_bwd<double, true>), dim3(blocks), dim3(kTile), 0, s, L, level);
        else hipLaunchKernelGGL((k_bwd<float, true>), dim3(blocks), dim3(kTile), 0, s, L, level);
    } else {
        if (fp64) hipLaunchKernelGGL((k_bwd<double, false>), dim3(blocks), dim3(kTile), 0, s, L, level);
        else hipLaunchKernelGGL((k_bwd<float, false>), dim3(blocks), dim3(kTile), 0, s, L, level);
    }
}
static size_t sub_lds(const SubLds &D, int entries, int index_bytes, bool fp64) {
    return (fp64 ? sizeof(d4) : sizeof(f4)) * (size_t)entries + sizeof(SubNode) * (size_t)D.nodes + (size_t)index_bytes +
           sizeof(int) * (size_t)(D.heights + 1);
}
template <typename T, bool Fused>
static void sub_fwd_of(hipStream_t s, LaunchSet L, int blocks, const SubLds &D, size_t lds) {
    if (D.block == kSubBlock) hipLaunchKernelGGL((k_sub_fwd<T, Fused, kSubBlock>), dim3(blocks), dim3(kSubBlock), lds, s, L, D);
    else if (Fused || D.block == 64) hipLaunchKernelGGL((k_sub_fwd<T, Fused, 64>), dim3(blocks), dim3(64), lds, s, L, D);
    else hipLaunchKernelGGL((k_sub_fwd<T, false, 128>), dim3(blocks), dim3(128), lds, s, L, D);
}
void launch_sub_fwd(hipStream_t s, LaunchSet L, int blocks, const SubLds &D, bool fused, bool fp64) {
    if (blocks <= 0) return;
    const size_t lds = sub_lds(D, D.fwd, (int)sizeof(int2) * D.fwd, fp64);
    if (fp64) fused ? sub_fwd_of<double, true>(s, L, blocks, D, lds) : sub_fwd_of<double, false>(s, L, blocks, D, lds);
    else fused ? sub_fwd_of<float, true>(s, L, blocks, D, lds) : sub_fwd_of<float, false>(s, L, blocks, D, lds);
}
template <typename T>
static void sub_bwd_of(hipStream_t s, LaunchSet L, int blocks, const SubLds &D, size_t lds) {
    if (D.block == kSubBlock) hipLaunchKernelGGL((k_sub_bwd<T, kSubBlock>), dim3(blocks), dim3(kSubBlock), lds, s, L, D);
    else if (D.block == 64) hipLaunchKernelGGL((k_sub_bwd<T, 64>), dim3(blocks), dim3(64), lds, s, L, D);
    else hipLaunchKernelGGL((k_sub_bwd<T, 128>), dim3(blocks), dim3(128), lds, s, L, D);
}
void launch_sub_bwd(hipStream_t s, LaunchSet L, int blocks, const SubLds &D, bool fp64) {
    if (blocks <= 0) return;
    const size_t lds = sub_lds(D, D.bwd, (int)sizeof(int) * D.off, fp64);
    if (fp64) sub_bwd_of<double>(s, L, blocks, D, lds);
    else sub_bwd_of<float>(s, L, blocks, D, lds);
}
void launch_energy(hipStream_t s, LaunchSet L, int blocks, bool fp64) {
    if (blocks <= 0) return;
    if (fp64) hipLaunchKernelGGL(k_energy<double>, dim3(blocks), dim3(kBlock), 0, s, L);
    else hipLaunchKernelGGL(k_energy<float>, dim3(blocks), dim3(kBlock), 0, s, L);
}

}  // namespace md

namespace md {
void set_error(const std::string &msg);
}

// Host diagnostic: the local step's rotation code compiled for the host (correctly rounded
// reciprocal and square roots instead of the device's approximate ones).
extern "C" int md_host_best_rotation(int fp64, int count, const double *cov, const double *prev, double *quat,
                                     int *fallback) {
    if (count < 0 || (count > 0 && (!cov || !quat))) {
        md::set_error("md_host_best_rotation: invalid argument");
        return MD_ERR_INVALID;
    }
    for (int k = 0; k < count; ++k) {
        const double *c = cov + 9 * (size_t)k;
        const double p[4] = {prev ? prev[4 * k] : 0.0, prev ? prev[4 * k + 1] : 0.0, prev ? prev[4 * k + 2] : 0.0,
                             prev ? prev[4 * k + 3] : 1.0};
        bool qcp;
        if (fp64) {
            double m[9], q[4];
            for (int i = 0; i < 9; ++i) m[i] = c[i];
            qcp = md::best_rotation<double>(m, p[0], p[1], p[2], p[3], q[0], q[1], q[2], q[3]);
            for (int i = 0; i < 4; ++i) quat[4 * k + i] = q[i];
        } else {
            float m[9], q[4];
            for (int i = 0; i < 9; ++i) m[i] = (float)c[i];
            qcp = md::best_rotation<float>(m, (float)p[0], (float)p[1], (float)p[2], (float)p[3], q[0], q[1], q[2], q[3]);
            for (int i = 0; i < 4; ++i) quat[4 * k + i] = q[i];
        }
        if (fallback) fallback[k] = qcp ? 0 : 1;
    }
    return MD_OK;
}
