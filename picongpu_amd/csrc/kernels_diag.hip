// Diagnostics of the PIC step on the device.
//
// Gauss-law residual eps0 * div E - rho at the cell origins in FP64, the
// quantity ChargeConservation::notify reports
// (plugins/ChargeConservation.tpp:181-260: backward-difference divergence
// `Div` :118-136, charge density from the particles' assignment shape). The
// charge density uses each species' ChargeAssignment B-spline evaluated in
// FP32 per axis and multiplied in FP64; it is accumulated with FP64 atomics,
// so the residual is reproducible to FP64 round-off (not bit for bit).
#include <array>
#include <mutex>

#include "pic_device.hpp"
#include "pic_kernels.hpp"

namespace pic {

// One block per supercell: its particles' charge is summed in an LDS tile of
// the supercell and the nodes around it, which is added to rho once. Adding
// every particle's nodes to rho directly (125 FP64 atomics each with PQS)
// took 711 us in a box of 48x40x44 cells and 6 particles a cell, the tile
// 56 us; most of that is the FP64 LDS additions.
template <int SUPP>
__global__ __launch_bounds__(256) void kChargeDensity(SpeciesDev S, GridDev g, double qScale, double* rho) {
    constexpr int begin = Shape<SUPP>::begin;
    // nodes begin .. begin + SUPP around a particle's cell
    constexpr int TX = SCX + SUPP, TY = SCY + SUPP, TZ = SCZ + SUPP, TV = TX * TY * TZ;
    __shared__ double tile[TV];
    int const sc = blockIdx.x;
    int const n = (int)S.count[sc];
    if (n == 0) return;  // uniform
    int const sx = sc % g.nscx;
    int const sy = (sc / g.nscx) % g.nscy;
    int const sz = sc / (g.nscx * g.nscy);
    size_t const base = slotBase(S, sc);
    for (int t = threadIdx.x; t < TV; t += blockDim.x) tile[t] = 0.0;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        size_t const gi = base + i;
        int const lc = S.cell[gi];
        double* const corner = tile + (lc % SCX) + TX * (((lc / SCX) % SCY) + TY * (lc / (SCX * SCY)));
        float const p[3] = {S.pos[0][gi], S.pos[1][gi], S.pos[2][gi]};
        double const q = (double)S.charge * (double)S.w[gi] * qScale;
        double wgt[3][SUPP + 1];
#pragma unroll
        for (int d = 0; d < 3; ++d)
#pragma unroll
            for (int o = 0; o <= SUPP; ++o) wgt[d][o] = (double)Shape<SUPP>::assign((float)(begin + o) - p[d]);
#pragma unroll
        for (int oz = 0; oz <= SUPP; ++oz)
#pragma unroll
            for (int oy = 0; oy <= SUPP; ++oy)
#pragma unroll
                for (int ox = 0; ox <= SUPP; ++ox) {
                    double const v = q * wgt[0][ox] * wgt[1][oy] * wgt[2][oz];
                    if (v != 0.0)
                        __hip_atomic_fetch_add(corner + (oz * TY + oy) * TX + ox, v, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < TV; t += blockDim.x) {
        double const v = tile[t];
        int xx = sx * SCX + begin + t % TX, yy = sy * SCY + begin + (t / TX) % TY, zz = sz * SCZ + begin + t / (TX * TY);
        if (v == 0.0 || outsideOpen(g, xx, yy, zz)) continue;
        xx = xx < 0 ? xx + g.nx : (xx >= g.nx ? xx - g.nx : xx);
        yy = yy < 0 ? yy + g.ny : (yy >= g.ny ? yy - g.ny : yy);
        zz = zz < 0 ? zz + g.nz : (zz >= g.nz ? zz - g.nz : zz);
        unsafeAtomicAdd(rho + (size_t)xx + (size_t)g.nx * ((size_t)yy + (size_t)g.ny * zz), v);
    }
}

__global__ __launch_bounds__(256) void kGaussResidual(FieldArgs a, double eps0, double* inout) {
    size_t const n = (size_t)a.g.nx * a.g.ny * a.g.nz;
    size_t const i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int const x = (int)(i % a.g.nx);
    int const y = (int)((i / a.g.nx) % a.g.ny);
    int const z = (int)(i / ((size_t)a.g.nx * a.g.ny));
    int const xm = x == 0 ? a.g.nx - 1 : x - 1;
    int const ym = y == 0 ? a.g.ny - 1 : y - 1;
    int const zm = z == 0 ? a.g.nz - 1 : z - 1;
    size_t const ix = (size_t)xm + (size_t)a.g.nx * ((size_t)y + (size_t)a.g.ny * z);
    size_t const iy = (size_t)x + (size_t)a.g.nx * ((size_t)ym + (size_t)a.g.ny * z);
    size_t const iz = (size_t)x + (size_t)a.g.nx * ((size_t)y + (size_t)a.g.ny * zm);
    // beyond an open border E reads zero
    double const ex = (a.g.open & 1) && x == 0 ? 0.0 : (double)a.E[0][ix];
    double const ey = (a.g.open & 2) && y == 0 ? 0.0 : (double)a.E[1][iy];
    double const ez = (a.g.open & 4) && z == 0 ? 0.0 : (double)a.E[2][iz];
    double div = ((double)a.E[0][i] - ex) / (double)a.cell[0];
    div += ((double)a.E[1][i] - ey) / (double)a.cell[1];
    div += ((double)a.E[2][i] - ez) / (double)a.cell[2];
    inout[i] = eps0 * div - inout[i];
}

__global__ __launch_bounds__(256) void kZeroD(double* p, size_t n) {
    size_t const i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// Scratch of the allocation-free Gauss residual: one FP64 value per cell,
// at most kNoAllocMaxCells cells. Each device holds its own copy for the
// life of the process; host code reaches it only through the address
// hipGetSymbolAddress returns on that device.
static __device__ __align__(256) double scratch[kNoAllocMaxCells];

hipError_t noAllocScratch(int device, double** out) {
    static std::mutex lock;
    static std::array<double*, kNoAllocMaxDevices> addr{};
    if (device < 0 || device >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> guard(lock);
    if (!addr[device]) {
        int current = 0;
        hipError_t e = hipGetDevice(&current);
        if (e != hipSuccess) return e;
        if (current != device) return hipErrorInvalidDevice;  // the caller makes `device` current
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        addr[device] = static_cast<double*>(p);
    }
    *out = addr[device];
    return hipSuccess;
}

hipError_t launchGaussResidual(const FieldArgs& f, const SpeciesDev* sp, const int* supp, int nsp, double qScale,
                               double eps0, double* buf, hipStream_t s) {
    size_t const n = (size_t)f.g.nx * f.g.ny * f.g.nz;
    int const nsc = f.g.nscx * f.g.nscy * f.g.nscz;
    hipLaunchKernelGGL(kZeroD, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, buf, n);
    for (int k = 0; k < nsp; ++k) {
        if (supp[k] == 2)
            hipLaunchKernelGGL(kChargeDensity<2>, dim3(nsc), dim3(256), 0, s, sp[k], f.g, qScale, buf);
        else if (supp[k] == 3)
            hipLaunchKernelGGL(kChargeDensity<3>, dim3(nsc), dim3(256), 0, s, sp[k], f.g, qScale, buf);
        else
            hipLaunchKernelGGL(kChargeDensity<4>, dim3(nsc), dim3(256), 0, s, sp[k], f.g, qScale, buf);
        hipError_t const e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kGaussResidual, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, f, eps0, buf);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The shortened FP32 operations against their IEEE values, mantissa by
// mantissa. The references are FP64 operations rounded to FP32: 53 bits are
// more than twice 24 and two, so the second rounding changes nothing.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void countDifferent(float a, float b, unsigned long long* bad) {
    bool const same = __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b);
    unsigned long long const m = __ballot(!same);
    if (m != 0ull && (threadIdx.x & 63) == 0) atomicAdd(bad, (unsigned long long)__popcll(m));
}

// every float of [2^e, 2^(e+1))
__global__ __launch_bounds__(256) void kCheckReciprocals(int e, unsigned long long* bad) {
    uint32_t const i = blockIdx.x * 256u + threadIdx.x;  // 2^23 threads
    float const x = __uint_as_float(((uint32_t)(127 + e) << 23) | i);
    float const inverse = (float)(1.0 / (double)x);
    if (e <= 64) countDifferent(recipOfRoot(x), inverse, bad);  // a root lies below 2^64
    if (e < 0) return;
    countDifferent(recipAbove1(x), inverse, bad + 1);
    countDifferent(sqrtAbove1(x), (float)sqrt((double)x), bad + 2);
}

// every mantissa and sign divided by c, the exponents spread over 2^-60 .. 2^59
__global__ __launch_bounds__(256) void kCheckDivExact(float c, unsigned long long* bad) {
    uint32_t const i = blockIdx.x * 256u + threadIdx.x;  // 2^24 threads
    uint32_t h = i * 2654435761u;
    h ^= h >> 15;
    h *= 2246822519u;
    h ^= h >> 13;
    float const x = __uint_as_float(((127u - 60u + h % 120u) << 23) | (i & 0x7fffffu) | (i >> 23 << 31));
    countDifferent(divExact(x, 1.0 / (double)c), (float)((double)x / (double)c), bad);
}

// zeros, infinities, NaN and the ends of the domains
__global__ __launch_bounds__(64) void kCheckSpecial(unsigned long long* bad) {
    float const inf = __uint_as_float(0x7f800000u), nan = __uint_as_float(0x7fc00000u);
    float const root[4] = {0.0f, inf, nan, 1.0f}, above1[4] = {inf, nan, 1.0f, 3.4028235e38f};
    float const r = root[threadIdx.x & 3], x = above1[threadIdx.x & 3];
    countDifferent(recipOfRoot(r), (float)(1.0 / (double)r), bad);
    countDifferent(recipAbove1(x), (float)(1.0 / (double)x), bad + 1);
    countDifferent(sqrtAbove1(x), (float)sqrt((double)x), bad + 2);
    float const q[4] = {0.0f, -0.0f, -inf, nan};
    countDifferent(divExact(q[threadIdx.x & 3], 1.0 / 1.7416), q[threadIdx.x & 3], bad + 3);
}

hipError_t launchArithmeticCheck(const float* divisors, int n, unsigned long long* bad, hipStream_t s) {
    for (int e = -75; e <= 127; ++e) hipLaunchKernelGGL(kCheckReciprocals, dim3(1u << 15), dim3(256), 0, s, e, bad);
    for (int k = 0; k < n; ++k) hipLaunchKernelGGL(kCheckDivExact, dim3(1u << 16), dim3(256), 0, s, divisors[k], bad + 3);
    hipLaunchKernelGGL(kCheckSpecial, dim3(1), dim3(64), 0, s, bad);
    return hipGetLastError();
}

}  // namespace pic
