// Whole small Dirichlet cubes in one block (gfx950): 15 x 15 planes, 15 or 31 of
// them.
//
// The three launches of such a solve (x and y transforms, z systems, transforms
// back) are each shorter than the host takes to launch it, and a batch moves the
// field through memory three times.  Here a block solves a problem with one read
// and one write:
//   1. a plane is transformed along x and y in LDS by the 32 lanes that loaded it;
//   2. a thread collects its mode's values from all planes into registers and
//      solves the z system there (cyclic reduction, every level local);
//   3. the planes go back through LDS, are transformed and stored by their lanes.
// Only the two exchanges between planes and modes need the block's barrier.
// Three launches / one, us a solve: 15^3 FP64 13.2 / 8.7, FP32 13.4 / 7.4, 512 of
// them 39.6 / 16.6 and 24.8 / 10.8; 15 x 15 x 31 FP64 13.6 / 13.7, FP32 13.5 / 9.7,
// 512 of them 55.5 / 32.3 and 40.9 / 20.0.  What bounds it is one CU's LDS and
// arithmetic: at 31 x 31 planes one problem takes 45 us and three launches 14, so
// those keep the launches.
#include <hip/hip_runtime.h>

#include "dst_device.hpp"
#include "kernel_util.hpp"
#include "kernels.hpp"

namespace fdmgpu {

template <typename T, int LOGZ>
struct SmallCfg {
    static constexpr int LOGN = 4;
    using S = DstShape<LOGN>;
    using Lane = DstLaneLds<T, LOGN>;
    static constexpr int N = 1 << LOGN, NZ = 1 << LOGZ, P = N + S::PAD, PL = N * P;
    static constexpr int LANES = N / 2 * S::N1;   // lanes per plane
    static constexpr int NT = NZ * LANES;
    static constexpr size_t lds_bytes() { return sizeof(T) * (size_t)(NZ * PL + Lane::kValues); }
    static_assert(NT % 64 == 0 && NT <= 1024 && N * N <= NT, "whole wavefronts, a thread per mode");
};

// The z system of one mode in one thread (see cr_level in dst_device.hpp), n =
// 2^Q - 1 rows; v[2^Q - 1] is scratch.  Operation for operation zcr_strip_kernel's in
// chunks of 16 rows, its default: of 31 rows the middle one separates two chunks,
// whose parts of its sum are added up apart.  (Explicit fma: else the scale of the
// right-hand side may be contracted into the first level's sum.)
template <int Q, typename T>
__device__ __forceinline__ void cr_column(T (&v)[1 << Q], const CrLevels<T, Q>& L) {
    constexpr int C = 1 << Q, SEP = C > 16 ? C / 2 - 1 : -1;
    static_assert(C <= 32, "at most two chunks");
    [[maybe_unused]] T below = T(0), above = T(0);
    static_for<1, Q>([&](auto ll) {
        constexpr int l = decltype(ll)::value, st = 1 << l, h = st >> 1;
#pragma unroll
        for (int r = st - 1; r < C - 1; r += st) {
            if (r == SEP) {
                below = fma(L.alpha[l], v[r - h], below);
                above = fma(L.alpha[l], v[r + h], above);
            } else {
                v[r] = fma(L.alpha[l], v[r - h] + v[r + h], v[r]);
            }
        }
    });
    if constexpr (SEP >= 0) v[SEP] = v[SEP] + below + above;
    v[C / 2 - 1] *= L.inv_d[Q - 1];
    v[C - 1] = T(0);
    static_for<1, Q>([&](auto ll) {
        constexpr int l = Q - decltype(ll)::value, st = 1 << l, h = st >> 1;
#pragma unroll
        for (int r = h - 1; r < C - 1; r += st) {
            const T left = r - h >= 0 ? v[r - h >= 0 ? r - h : 0] : T(0);
            v[r] = fma(-L.c[l - 1], left + v[r + h], v[r]) * L.inv_d[l - 1];
        }
    });
}

// The z systems in double (FP32 plans too, as zcr_kernel).  (fx, fy), (ix, iy):
// scales of the forward and inverse transforms.
template <typename T, int LOGZ>
__global__ __launch_bounds__((SmallCfg<T, LOGZ>::NT)) void small_cube_kernel(
    const BatchPtr<const T> in, const BatchPtr<T> out, const T fx, const T fy, const T ix, const T iy,
    const T* __restrict__ tables, const T* __restrict__ lmx, const T* __restrict__ lmy, const double b,
    const double gamma) {
    using C = SmallCfg<T, LOGZ>;
    using IO = PencilIO<kDst, C::LOGN>;
    using LX = PlaneLayout<C::P, C::S::N1, true>;
    using LY = PlaneLayout<C::P, C::S::N1, false>;
    constexpr int N = C::N, n = N - 1, nz = C::NZ - 1, LANES = C::LANES;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* const lds = reinterpret_cast<T*>(smem_raw);
    T* const consts = lds + C::NZ * C::PL;
    const int tid = threadIdx.x, li = tid % LANES, z = tid / LANES;
    T* const plane = lds + z * C::PL;   // plane nz is a dummy, all zeros
    const auto src = as_global(in(blockIdx.x));
    const auto dst = as_global(out(blockIdx.x));
    // lane (x, y0) of a plane loads and stores rows y0, y0 + STEP, ...
    constexpr int STEP = LANES / N, ROWS = N / STEP;
    const int x = li % N, y0 = li / N;
    auto on = [&](int y) { return x < n && y < n && z < nz; };
    T v[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) v[i] = on(y0 + STEP * i) ? src[(z * n + y0 + STEP * i) * n + x] : T(0);
    C::Lane::fill(tables, consts, tid, C::NT);
    typename C::Lane L;
    L.init(consts, tid & (C::S::N1 - 1));
    if (li < N) {   // dummy row and column (the transforms leave them 0)
        plane[LX::at(0, li)] = T(0);
        plane[LX::at(li, 0)] = T(0);
    }
    const int kx = tid % N, ky = tid / N;
    const bool mode = kx < n && ky < n;
    const double lam = mode ? (double)lmx[kx] + (double)lmy[ky] : 1.0;
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
        if (x < n && y0 + STEP * i < n) plane[LX::at(y0 + STEP * i + 1, x + 1)] = v[i];
    __syncthreads();
    // (each pass computes its addresses anew: shared they would be held in
    // registers the z systems need)
    auto passes = [&](const T sx, const T sy) {
        pencil_pairs<kDst, T, C::LOGN, N / 2, LX, LANES, typename C::Lane>(plane, L, sx, opaque_volatile(li));
        pencil_pairs<kDst, T, C::LOGN, N / 2, LY, LANES, typename C::Lane>(plane, L, sy, opaque_volatile(li));
    };
    passes(fx, fy);
    __syncthreads();
    double g[C::NZ];
    if (mode) {
#pragma unroll
        for (int k = 0; k < C::NZ; ++k) g[k] = (double)lds[k * C::PL + LX::at(IO::out(ky), IO::out(kx))] * gamma;
        CrLevels<double, LOGZ> cr;
        cr_levels<double, LOGZ>(cr, b, lam);
        cr_column<LOGZ>(g, cr);
    }
    __syncthreads();   // outputs sit permuted: a mode's slot to write is another's to read
    if (mode) {
#pragma unroll
        for (int k = 0; k < C::NZ; ++k) lds[k * C::PL + LX::at(ky + 1, kx + 1)] = (T)g[k];
    }
    __syncthreads();
    passes(ix, iy);
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
        if (on(y0 + STEP * i)) dst[(z * n + y0 + STEP * i) * n + x] = plane[LX::at(IO::out(y0 + STEP * i), IO::out(x))];
}

template <typename T, int LOGZ>
static hipError_t small_k(const SmallCubeArgs& a) {
    using C = SmallCfg<T, LOGZ>;
    auto k = small_cube_kernel<T, LOGZ>;
    const hipError_t e = allow_lds(k, C::lds_bytes());
    if (e != hipSuccess) return e;
    const BatchPtr<const T> in{(const T*)a.in, a.in_tab, a.bs};
    const BatchPtr<T> out{(T*)a.out, a.out_tab, a.bs};
    hipLaunchKernelGGL(k, dim3(a.batch), dim3(C::NT), C::lds_bytes(), a.stream, in, out, (T)a.fx, (T)a.fy, (T)a.ix,
                       (T)a.iy, (const T*)a.tables, (const T*)a.lmx, (const T*)a.lmy, a.b, a.gamma);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_small_cube(int logn, int logz, const SmallCubeArgs& a) {
    if (logn == 4 && logz == 4) return small_k<T, 4>(a);
    if (logn == 4 && logz == 5) return small_k<T, 5>(a);
    return hipErrorInvalidValue;
}

bool small_cube_ok(int logn, int logz) { return logn == 4 && (logz == 4 || logz == 5); }

template hipError_t launch_small_cube<float>(int, int, const SmallCubeArgs&);
template hipError_t launch_small_cube<double>(int, int, const SmallCubeArgs&);

}  // namespace fdmgpu
