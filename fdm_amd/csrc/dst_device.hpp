// Device building blocks for the fast Poisson solve on gfx950 (CDNA4, wave64).
//
//  * dft<R>:        forward DFT of R <= 32 complex values held in registers
//                   (fully unrolled radix-2, compile-time twiddles).
//  * dst_pairs<>:   DST-I of pencils held in LDS, two pencils per job.
//
// DST-I definition (the transform FFT<T>::sFFT computes, reference
// src/fft.cpp:293-365):  X[k] = scale * sum_{j=1}^{N-1} x[j] sin(pi j k / N),
// k = 1..N-1, N = 2^LOGN.  Algorithm (not the reference's Samarskii-Nikolaev
// recursion, which is sequential per pencil):
//   1. w_j = sin(pi j/N)(x_j + x_{N-j}) + (x_j - x_{N-j})/2        (w_0 = 0)
//          = (sin(pi j/N) + 1/2)(x_j + x_{N-j}) - x_{N-j}   (one add, one fma)
//      Two pencils a, b are packed as z_j = w^a_j + i w^b_j.
//   2. Z = FFT_N(z), done as a 4-step FFT N = N1 x N2: N1 lanes per job each
//      run an N2-point DFT in registers, twiddle by w_N^{j1 k2}, exchange
//      through the pencils' own LDS slots, then N1-point DFTs.
//   3. With W = the real DFT of w:  Re W_k = X_{2k+1} - X_{2k-1},
//      Im W_k = -X_{2k}.  So X_{2k} comes directly and the odd outputs are a
//      prefix sum X_{2k+1} = Re W_0 / 2 + sum_{i=1..k} Re W_i, computed as a
//      per-lane running sum plus a shuffle scan across the job's N1 lanes.
// Everything happens in place in the pencils' N LDS slots (slot 0 is a
// dummy that reads as zero after the transform), so an N x N plane (one
// dummy row, one dummy column) holds a full 127^2 FP64 plane in 139 KB.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.hpp"   // kDst, kRdftFwd, kRdftInv

namespace fdmgpu {

constexpr int ilog2(int v) { return v <= 1 ? 0 : 1 + ilog2(v >> 1); }
constexpr int bitrev(int v, int bits) {
    int r = 0;
    for (int b = 0; b < bits; b++)
        if (v & (1 << b)) r |= 1 << (bits - 1 - b);
    return r;
}

// cos(2 pi m / 32) from the first quadrant by symmetry (exact zeros).
constexpr double kQuarter[9] = {1.0,
                                0.98078528040323044912618223613424,
                                0.92387953251128675612818318939679,
                                0.83146961230254523707878837761791,
                                0.70710678118654752440084436210485,
                                0.55557023301960222474283081394853,
                                0.38268343236508977172845998403040,
                                0.19509032201612826784828486847702,
                                0.0};
constexpr double cos32(int m) {
    m = ((m % 32) + 32) % 32;
    return m <= 8 ? kQuarter[m] : m <= 16 ? -kQuarter[16 - m] : m <= 24 ? -kQuarter[m - 16] : kQuarter[32 - m];
}
constexpr double sin32(int m) { return cos32(m - 8); }

// Butterfly (a, b) <- (a + w b, a - w b), w = exp(-2 pi i K / L), L | 32, all
// compile time.  Every product feeds an explicit fma (6 operations where w is
// neither 1 nor -i, 8 as a product and two sums), which also leaves the
// compiler no choice of which product to contract: the same transform gives the
// same bits in every kernel.
template <int L, int K, typename T>
__device__ __forceinline__ void butterfly(T& ar, T& ai, T& br, T& bi) {
    static_assert(0 <= K && 2 * K < L, "first half turn");
    if constexpr (K == 0) {
        const T r = ar - br, i = ai - bi;
        ar += br;
        ai += bi;
        br = r;
        bi = i;
    } else if constexpr (4 * K == L) {   // w = -i
        const T r = ar - bi, i = ai + br;
        ar += bi;
        ai -= br;
        br = r;
        bi = i;
    } else if constexpr (8 * K == L || 8 * K == 3 * L) {   // w = +-sqrt(1/2) - i sqrt(1/2)
        constexpr T h = (T)kQuarter[4];
        const T d = 8 * K == L ? br + bi : bi - br, e = 8 * K == L ? bi - br : -(br + bi);
        br = fma(-h, d, ar);
        bi = fma(-h, e, ai);
        ar = fma(h, d, ar);
        ai = fma(h, e, ai);
    } else {
        constexpr int m = K * (32 / L);
        constexpr T c = (T)cos32(m);
        constexpr T s = (T)(-sin32(m));
        const T r = fma(-s, bi, fma(c, br, ar)), i = fma(c, bi, fma(s, br, ai));
        br = fma(T(2), ar, -r);
        bi = fma(T(2), ai, -i);
        ar = r;
        ai = i;
    }
}

// (re, im) *= c + i s
template <typename T>
__device__ __forceinline__ void rotate(T& re, T& im, const T c, const T s) {
    const T r = fma(-s, im, c * re), i = fma(c, im, s * re);
    re = r;
    im = i;
}

// In-register forward DFT of size R (natural order in and out).
template <int R, typename T>
__device__ __forceinline__ void dft(T (&re)[R], T (&im)[R]) {
    static_assert(R >= 1 && R <= 32 && (R & (R - 1)) == 0, "radix");
    if constexpr (R > 1) {
        constexpr int LOG = ilog2(R);
        static_for<0, R>([&](auto ii) {
            constexpr int i = decltype(ii)::value;
            constexpr int r = bitrev(i, LOG);
            if constexpr (i < r) {
                T t = re[i];
                re[i] = re[r];
                re[r] = t;
                t = im[i];
                im[i] = im[r];
                im[r] = t;
            }
        });
        static_for<1, LOG + 1>([&](auto ss) {
            constexpr int len = 1 << decltype(ss)::value;
            static_for<0, R / len>([&](auto bb) {
                static_for<0, len / 2>([&](auto kk) {
                    constexpr int a = decltype(bb)::value * len + decltype(kk)::value;
                    constexpr int b = a + len / 2;
                    butterfly<len, decltype(kk)::value>(re[a], im[a], re[b], im[b]);
                });
            });
        });
    }
}

template <int LOGN>
struct DstShape {
    static constexpr int N = 1 << LOGN;
    static constexpr int N1 = 1 << (LOGN / 2);   // lanes per job
    static constexpr int N2 = N / N1;            // N2 >= N1
    static constexpr int M = N / 2;
    static constexpr int KC = M / N1;            // post-processing outputs per lane (>= 1)
    static constexpr int LOGKC = ilog2(KC);
    // LDS padding: a pencil-to-pencil stride congruent to N1 mod 32 banks spreads
    // the N1 lanes of neighbouring jobs over distinct banks.
    static constexpr int PAD = N1;

    // Slot of the step-1 result Y[j1][k2] (XOR swizzle: conflict-free for the
    // step-1 stores, contiguous in j1, and the step-2 loads, contiguous in k2).
    __device__ static constexpr int posY(int j1, int k2) { return N1 * k2 + (j1 ^ (k2 & (N1 - 1))); }
    // Slot of the FFT output Z_k (swizzled so step 3's per-lane k ranges hit
    // distinct banks).
    __device__ static constexpr int posZ(int k) {
        return KC > 1 ? ((k & ~(KC - 1)) | ((k ^ (k >> LOGKC)) & (KC - 1))) : k;
    }
    // Slot that receives the transform output X_j.  Pencils are independent, so
    // the outputs may sit in any fixed permutation between passes.  Step 3's
    // lane t writes j = N2*t + c (c fixed per store), so XOR-ing the low bits of
    // j with t makes those stores hit distinct banks, while runs of consecutive
    // j stay conflict-free for the natural-order reads.  sigma is an
    // involution and sigma(0) = 0.
    static constexpr int LOGN2 = ilog2(N2);
    __device__ static constexpr int sigma(int j) { return j ^ ((j >> LOGN2) & (N1 - 1)); }
};

// Per-lane constants of the DST (the lane's index t inside its job is fixed for
// the whole kernel): twiddles w_N^{t k2}, k2 < N2, and shifted sines
// sin(pi (t+N1 j2)/N) + 1/2.
template <typename T, int LOGN>
struct DstLane {
    using S = DstShape<LOGN>;
    T twr[S::N2], twi[S::N2], sp[S::N2];
    // tables (global memory): cos(2 pi m/N), -sin(2 pi m/N), sin(pi m/N) + 1/2, m < N
    __device__ __forceinline__ void init(const T* __restrict__ tables, const int t) {
        constexpr int N = S::N, N1 = S::N1, N2 = S::N2;
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) {
            twr[k2] = tables[t * k2];
            twi[k2] = tables[N + t * k2];
            sp[k2] = tables[2 * N + t + N1 * k2];
        }
    }
    __device__ __forceinline__ T sine(const int j2) const { return sp[j2]; }
    __device__ __forceinline__ void twiddle(const int k2, T& c, T& s) const {
        c = twr[k2];
        s = twi[k2];
    }
};

// The same constants with the shifted sines read from a per-block LDS copy of
// the table at each use instead of held in registers (N2 registers of T fewer
// per lane): for kernels whose register budget is taken by other work.
template <typename T, int LOGN>
struct DstLaneLdsSine {
    using S = DstShape<LOGN>;
    T twr[S::N2], twi[S::N2];
    const T* sl;   // LDS: sin(pi m/N) + 1/2, m < N, from the lane's own m = t
    // lds_sines: N values of the block's LDS, filled by fill_sines before the
    // first barrier
    __device__ __forceinline__ void init(const T* __restrict__ tables, const T* lds_sines, const int t) {
        constexpr int N = S::N, N2 = S::N2;
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) {
            twr[k2] = tables[t * k2];
            twi[k2] = tables[N + t * k2];
        }
        sl = lds_sines + t;
    }
    __device__ static void fill_sines(const T* __restrict__ tables, T* lds_sines, const int tid, const int nt) {
        for (int m = tid; m < S::N; m += nt) lds_sines[m] = tables[2 * S::N + m];
    }
    __device__ __forceinline__ T sine(const int j2) const { return sl[S::N1 * j2]; }
    __device__ __forceinline__ void twiddle(const int k2, T& c, T& s) const {
        c = twr[k2];
        s = twi[k2];
    }
};

// All the constants from LDS: the shifted sines as above, the twiddles from a
// copy laid out [k2][t] as (re, im) pairs, so a job's lanes read consecutive
// pairs.  For kernels that hold data in registers through a pass.
template <typename T, int LOGN>
struct DstLaneLds {
    using S = DstShape<LOGN>;
    static constexpr int kValues = S::N + 2 * S::N1 * S::N2;   // values of T in LDS (8-byte aligned for float)
    const T* sl;
    const T* tl;
    __device__ __forceinline__ void init(const T* lds, const int t) {
        sl = lds + t;
        tl = lds + S::N + 2 * t;
    }
    __device__ static void fill(const T* __restrict__ tables, T* lds, const int tid, const int nt) {
        for (int m = tid; m < S::N; m += nt) lds[m] = tables[2 * S::N + m];
        for (int m = tid; m < S::N1 * S::N2; m += nt) {
            const int k2 = m / S::N1, t = m % S::N1;
            lds[S::N + 2 * m] = tables[t * k2];
            lds[S::N + 2 * m + 1] = tables[S::N + t * k2];
        }
    }
    __device__ __forceinline__ T sine(const int j2) const { return sl[S::N1 * j2]; }
    __device__ __forceinline__ void twiddle(const int k2, T& c, T& s) const {
        c = tl[2 * S::N1 * k2];
        s = tl[2 * S::N1 * k2 + 1];
    }
};

// LDS layouts of a set of pencils.  Measured on gfx950: b32 accesses and b64
// reads see 32 banks per half-wavefront (b64 reads in 8-byte banks), b64
// writes 16 eight-byte banks per quarter-wavefront.  A job's N1 lanes touch N1
// slots that are distinct mod N1, so a row pitch congruent to N1 mod 32 makes
// row-pencil (x) accesses conflict-free.  Column-pencil (y) accesses are then
// spread by shifting each row by f(row) < N1 slots (the pitch leaves room).
// The shift is additive rather than an XOR so that, for a fixed row, slot
// offsets stay compile-time constants a ds instruction can carry.
template <int N1>
struct RowSwizzle {
    static constexpr int QJ = 32 / N1;                            // jobs per half-wavefront
    static constexpr int LS = ilog2(QJ);
    static constexpr int FM = (N1 * N1 > 32) ? (N1 * N1) / 32 - 1 : 0;
    static constexpr int FMAX = FM << LS;                         // largest f value
    __device__ static constexpr int f(int row) { return ((row >> LS) & FM) << LS; }
};

// Hides a value's derivation from the optimizer (no instruction is emitted).
__device__ __forceinline__ int opaque(int x) {
    asm("" : "+v"(x));
    return x;
}

// The same for a value computed anew where it stands (never hoisted or shared).
__device__ __forceinline__ int opaque_volatile(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// Plane of rows with pitch P; element (row, col) at row*P + col + f(row).
// Pencils are rows (x pass) or columns (y pass).
template <int P, int N1, bool ALONG_X>
struct PlaneLayout {
    using Sw = RowSwizzle<N1>;
    // pencil of job jj, and the distance to its second pencil: jobs in
    // order, pencils jj and jj + JOBS
    __device__ static constexpr int pencil(int jj) { return jj; }
    static constexpr int pair_delta(int jobs) { return jobs; }
    __device__ static constexpr int at(int row, int col) { return row * P + col + Sw::f(row); }
    __device__ static constexpr int addr(int pencil, int slot) {
        return ALONG_X ? at(pencil, slot) : at(slot, pencil);
    }
    // addr(pencil + DP, lv + cp) for a lane-dependent pencil and lv and
    // compile-time DP and cp, cp a multiple of N1.  f() has period N1 (it reads
    // only bits below log2(N1)), so f(lv + cp) = f(lv), and likewise
    // f(pencil + DP) = f(pencil) when N1 divides DP: the constant parts then
    // become an offset the ds instruction carries, and the lane part is
    // computed once per distinct (pencil, lv).  The lane part goes through
    // opaque() so the compiler cannot fold the constants back into the
    // row multiply.
    template <int DP>
    __device__ static int addr_split(int pencil, int lv, int cp) {
        if constexpr (ALONG_X) {
            if constexpr (DP % N1 == 0 || Sw::FM == 0)
                return opaque(pencil * P + Sw::f(pencil) + lv) + (DP * P + cp);
            else
                return opaque((pencil + DP) * P + Sw::f(pencil + DP) + lv) + cp;
        } else {
            return opaque(lv * P + Sw::f(lv) + pencil) + (DP + cp * P);
        }
    }
};

// v from lane - D within the lane's row of 16 (DPP row_shr:D, a VALU move:
// no LDS instruction as a shuffle through ds_bpermute would take); lanes
// whose source falls outside the row get v back.
template <int D, typename T>
__device__ __forceinline__ T row_shr(T v) {
    static_assert(D >= 1 && D <= 15, "row_shr range");
    if constexpr (sizeof(T) == 8) {
        const long long b = __builtin_bit_cast(long long, v);
        const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, 0x110 + D, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), 0x110 + D, 0xf, 0xf, false);
        return __builtin_bit_cast(T, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
    } else {
        const int b = __builtin_bit_cast(int, v);
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(b, b, 0x110 + D, 0xf, 0xf, false));
    }
}

// Inclusive scan across `width` consecutive lanes (width a power of two <= 64).
// Within a row of 16 lanes (width <= 16) the lane - d values come by DPP;
// a lane takes one only when lane - d is in its own group (t >= d), so the
// row_shr values from the neighbouring group are never used.
template <int WIDTH, typename T>
__device__ __forceinline__ T lane_scan_incl(T v) {
    if constexpr (WIDTH <= 16) {
        const int t = threadIdx.x & (WIDTH - 1);
        if constexpr (WIDTH > 1) {
            const T o = row_shr<1>(v);
            if (t >= 1) v += o;
        }
        if constexpr (WIDTH > 2) {
            const T o = row_shr<2>(v);
            if (t >= 2) v += o;
        }
        if constexpr (WIDTH > 4) {
            const T o = row_shr<4>(v);
            if (t >= 4) v += o;
        }
        if constexpr (WIDTH > 8) {
            const T o = row_shr<8>(v);
            if (t >= 8) v += o;
        }
    } else {
#pragma unroll
        for (int d = 1; d < WIDTH; d <<= 1) {
            T o = __shfl_up(v, d, WIDTH);
            if ((threadIdx.x & (WIDTH - 1)) >= d) v += o;
        }
    }
    return v;
}

// v of another lane by DPP control CTRL, 0 where that lane is none or the row
// of 16 is not in ROWS.
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T dpp_or_zero(T v) {
    if constexpr (sizeof(T) == 8) {
        const long long b = __builtin_bit_cast(long long, v);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
        return __builtin_bit_cast(T, (long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROWS, 0xf, false));
    }
}

// v of the lane's neighbour t ^ 1 (quad_perm 1, 0, 3, 2).
template <typename T>
__device__ __forceinline__ T lane_xor1(T v) {
    return dpp_or_zero<0xb1, 0xf>(v);
}

// Inclusive scan over each row (L = 16), half (32) or all (64) of the wavefront:
// rows of 16 by row_shr, then lane 15's sum into the next row (rows 1 and 3) and lane
// 31's into rows 2 and 3.
template <int L, typename T>
__device__ __forceinline__ T wave_scan_incl(T v) {
    v += dpp_or_zero<0x111, 0xf>(v);
    v += dpp_or_zero<0x112, 0xf>(v);
    v += dpp_or_zero<0x114, 0xf>(v);
    v += dpp_or_zero<0x118, 0xf>(v);
    if constexpr (L >= 32) v += dpp_or_zero<0x142, 0xa>(v);
    if constexpr (L == 64) v += dpp_or_zero<0x143, 0xc>(v);
    return v;
}

// Orders the LDS accesses of one wavefront across lanes.  A job's lanes lie in
// one wavefront, whose LDS instructions execute in issue order, so only the
// compiler's code motion has to be fenced.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Pencil transform kinds.
//   kDst:     DST-I, FFT<T>::sFFT (reference src/fft.cpp:293-365); N-1 points
//             in slots 1..N-1 (slot 0 is a dummy).
//   kRdftFwd: half-complex real DFT, FFT<T>::pFFT_1 (src/fft.cpp:108-193):
//             X[0] = s*sum x_j, X[k] = s*sum x_j cos(2 pi k j/N),
//             X[N-k] = s*sum x_j sin(2 pi k j/N) (0 < k < N/2),
//             X[N/2] = s*sum (-1)^j x_j; N points in slots 0..N-1.
//   kRdftInv: its inverse series, FFT<T>::pFFT (src/fft.cpp:195-212):
//             x_j = s*(X[0]/2 + X[N/2](-1)^j/2
//                   + sum_{0<k<N/2} X[k] cos(2 pi k j/N) + X[N-k] sin(2 pi k j/N)).
// pFFT(pFFT_1(x)) = (N/2) x, the same round-trip factor as the DST-I.

template <int KIND, int LOGN>
struct PencilIO {
    using S = DstShape<LOGN>;
    static constexpr int N = S::N;
    static constexpr int n = KIND == kDst ? N - 1 : N;   // points per pencil
    static constexpr int off = KIND == kDst ? 1 : 0;     // slot of point 0 on input
    // slot that holds output point m (0 <= m < n) after the transform
    __device__ static constexpr int out(int m) { return KIND == kDst ? S::sigma(m + 1) : S::posZ(m); }
};

// Transform of 2*JOBS pencils in LDS: pencil p, slot j at lds[Lay::addr(p, j)];
// job g transforms pencils g and g + JOBS (packed as the real and imaginary
// parts of one complex FFT of length N).  On entry the points sit in natural
// order from slot PencilIO::off (kDst: slot 0 holds a finite value); on exit
// output point m sits in slot PencilIO::out(m), times `scale` (kDst: slot 0
// holds 0).  All NT threads of the block call this; no block barrier inside
// (jobs never straddle a wavefront).
//
// kRdftFwd: Z = FFT(a + i b); A_k = (Z_k + conj Z_{N-k})/2,
//   B_k = (Z_k - conj Z_{N-k})/(2i), X_a[k] = Re A_k, X_a[N-k] = -Im A_k.
//   Step 3 reads Z_k, Z_{N-k} and writes X[k], X[N-k] into the same two slots.
// kRdftInv: C_k = X[k]/2 - i X[N-k]/2 (Hermitian; C_0, C_{N/2} real),
//   w = C^a + i C^b, x^a + i x^b = sum_k w_k e^{+2 pi i jk/N}
//   = conj(FFT(conj w)); step 2 writes the result directly.
template <int KIND, typename T, int LOGN, int JOBS, typename Lay, int NT, typename Lane = DstLane<T, LOGN>>
__device__ __forceinline__ void pencil_pairs(T* __restrict__ lds, const Lane& L, const T scale,
                                             const int tid) {
    using S = DstShape<LOGN>;
    constexpr int N = S::N, N1 = S::N1, N2 = S::N2, KC = S::KC;
    constexpr int WORK = JOBS * N1;
    static_assert(NT % N1 == 0 && 64 % N1 == 0, "jobs must not straddle wavefronts");
    const int t = tid & (N1 - 1);
#pragma unroll 1
    for (int base = 0; base < WORK; base += NT) {
        const int w = base + tid;
        if (w < WORK) {
            const int g = Lay::pencil(w / N1);
// slot = lv + cp: lv lane-dependent, cp a compile-time multiple of N1 (see
// PlaneLayout::addr_split); pencil gb = g + Lay::pair_delta(JOBS) sits at a constant offset
#define PA(lv, cp) lds[Lay::template addr_split<0>(g, (lv), (cp))]
#define PB(lv, cp) lds[Lay::template addr_split<Lay::pair_delta(JOBS)>(g, (lv), (cp))]

            // ---- step 1: pre-processing + N2-point DFTs over j2 (j = t + N1*j2)
            T yr[N2], yi[N2];
            const int tn0 = (N - t) & (N - 1);   // slot N - j for j = t (0 for j = 0)
#pragma unroll
            for (int j2 = 0; j2 < N2; ++j2) {
                const int j = t + N1 * j2;
                if constexpr (KIND == kRdftFwd) {
                    yr[j2] = PA(t, N1 * j2);
                    yi[j2] = PB(t, N1 * j2);
                } else {
                    // N - j = (N1 - t) + (N - N1 - N1*j2) for j2 > 0
                    const int jl = j2 == 0 ? tn0 : N1 - t, jc = j2 == 0 ? 0 : N - N1 - N1 * j2;
                    const T a0 = PA(t, N1 * j2), a1 = PA(jl, jc);
                    const T b0 = PB(t, N1 * j2), b1 = PB(jl, jc);
                    if constexpr (KIND == kDst) {
                        const T s = L.sine(j2);
                        yr[j2] = fma(s, a0 + a1, -a1);
                        yi[j2] = fma(s, b0 + b1, -b1);
                    } else if (2 * j2 < N2) {   // 0 <= j < N/2
                        const bool edge = j == 0;
                        yr[j2] = edge ? T(0.5) * a0 : T(0.5) * (a0 + b1);
                        yi[j2] = edge ? T(-0.5) * b0 : T(0.5) * (a1 - b0);
                    } else {                              // N/2 <= j < N
                        const bool edge = j == N / 2;
                        yr[j2] = edge ? T(0.5) * a0 : T(0.5) * (a1 - b0);
                        yi[j2] = edge ? T(-0.5) * b0 : T(-0.5) * (a0 + b1);
                    }
                }
            }
            dft<N2>(yr, yi);
#pragma unroll
            for (int k2 = 1; k2 < N2; ++k2) {
                T c, s;
                L.twiddle(k2, c, s);
                rotate(yr[k2], yi[k2], c, s);
            }
            wave_lds_sync();
#pragma unroll
            for (int k2 = 0; k2 < N2; ++k2) {   // posY(t, k2) = N1*k2 + (t ^ (k2 mod N1))
                const int lv = t ^ (k2 & (N1 - 1));
                PA(lv, N1 * k2) = yr[k2];
                PB(lv, N1 * k2) = yi[k2];
            }
            wave_lds_sync();

            // ---- step 2: N1-point DFTs over j1 for k2 = t + N1*r
            constexpr int RR = N2 / N1;
            T zr[N2], zi[N2];
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                T vr[N1], vi[N1];
#pragma unroll
                for (int j1 = 0; j1 < N1; ++j1) {   // posY(j1, k2) = N1*t + (j1 ^ t) + N1*N1*r
                    const int lv = N1 * t + (j1 ^ t);
                    vr[j1] = PA(lv, N1 * N1 * r);
                    vi[j1] = PB(lv, N1 * N1 * r);
                }
                dft<N1>(vr, vi);
#pragma unroll
                for (int k1 = 0; k1 < N1; ++k1) {
                    zr[r * N1 + k1] = vr[k1];
                    zi[r * N1 + k1] = vi[k1];
                }
            }
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < RR; ++r) {
#pragma unroll
                for (int k1 = 0; k1 < N1; ++k1) {
                    // posZ permutes aligned blocks of KC <= N1 slots, so
                    // posZ(t + cz) - cz < N1 for the multiple of N1 cz
                    const int cz = N1 * r + N2 * k1;
                    const int lv = S::posZ(t + cz) - cz;
                    if constexpr (KIND == kRdftInv) {   // x^a = Re Y, x^b = -Im Y
                        PA(lv, cz) = zr[r * N1 + k1] * scale;
                        PB(lv, cz) = -zi[r * N1 + k1] * scale;
                    } else {
                        PA(lv, cz) = zr[r * N1 + k1];
                        PB(lv, cz) = zi[r * N1 + k1];
                    }
                }
            }
            wave_lds_sync();

            if constexpr (KIND == kRdftFwd) {
                // ---- step 3: split the packed spectra; lane t owns k in [t*KC, (t+1)*KC)
                // and their mirrors N-k (k = 0: the Nyquist slot N/2)
#pragma unroll
                for (int i = 0; i < KC; ++i) {
                    const int k = t * KC + i;
                    const bool k0 = k == 0;
                    const int pk = S::posZ(k), pn = S::posZ(k0 ? N / 2 : N - k);
                    const T zkr = PA(pk, 0), zki = PB(pk, 0);
                    const T znr = PA(pn, 0), zni = PB(pn, 0);
                    PA(pk, 0) = (k0 ? zkr : T(0.5) * (zkr + znr)) * scale;
                    PB(pk, 0) = (k0 ? zki : T(0.5) * (zki + zni)) * scale;
                    PA(pn, 0) = (k0 ? znr : T(0.5) * (zni - zki)) * scale;
                    PB(pn, 0) = (k0 ? zni : T(0.5) * (zkr - znr)) * scale;
                }
                wave_lds_sync();
            } else if constexpr (KIND == kDst) {
                // ---- step 3: even outputs directly, odd outputs by prefix sum.
                // The 1/2 of both formulas is applied with the scale at the
                // store (a power of two: the results are bitwise the same).
                const T hs = T(0.5) * scale;
                T ae[KC], ao[KC], be[KC], bo[KC];
                T runA = T(0), runB = T(0);
#pragma unroll
                for (int i = 0; i < KC; ++i) {
                    const int k = t * KC + i;
                    const int pk = S::posZ(k), pn = S::posZ((N - k) & (N - 1));
                    const T zkr = PA(pk, 0), zki = PB(pk, 0);
                    const T znr = PA(pn, 0), zni = PB(pn, 0);
                    ae[i] = zni - zki;
                    be[i] = zkr - znr;
                    T dA = zkr + znr;
                    T dB = zki + zni;
                    if (k == 0) {
                        dA *= T(0.5);
                        dB *= T(0.5);
                    }
                    runA += dA;
                    runB += dB;
                    ao[i] = runA;
                    bo[i] = runB;
                }
                if constexpr (N1 > 1) {
                    const T offA = lane_scan_incl<N1>(runA) - runA;
                    const T offB = lane_scan_incl<N1>(runB) - runB;
#pragma unroll
                    for (int i = 0; i < KC; ++i) {
                        ao[i] += offA;
                        bo[i] += offB;
                    }
                }
                wave_lds_sync();
#pragma unroll
                for (int i = 0; i < KC; ++i) {
                    // sigma(2k + e) = t*N2 + ((2i + e) ^ t) for k = t*KC + i (2i + e < N2, t < N1):
                    // lane part t*N2 + (((2i + e) mod N1) ^ t), the rest a multiple of N1
                    const int k = t * KC + i;
                    const T e_a = k == 0 ? T(0) : ae[i] * hs;
                    const T e_b = k == 0 ? T(0) : be[i] * hs;
                    const int me = 2 * i, mo = 2 * i + 1;
                    const int le = t * N2 + ((me & (N1 - 1)) ^ t), lo = t * N2 + ((mo & (N1 - 1)) ^ t);
                    PA(le, me & ~(N1 - 1)) = e_a;
                    PB(le, me & ~(N1 - 1)) = e_b;
                    PA(lo, mo & ~(N1 - 1)) = ao[i] * hs;
                    PB(lo, mo & ~(N1 - 1)) = bo[i] * hs;
                }
                wave_lds_sync();
            }
#undef PA
#undef PB
        }
    }
}

template <typename T, int LOGN, int JOBS, typename Lay, int NT>
__device__ __forceinline__ void dst_pairs(T* __restrict__ lds, const DstLane<T, LOGN>& L, const T scale,
                                          const int tid) {
    pencil_pairs<kDst, T, LOGN, JOBS, Lay, NT>(lds, L, scale, tid);
}

// The DST of the rows (COLS false: PlaneLayout<P, 8, true>) or the columns
// (COLS true: PlaneLayout<P, 8, false>) of a 128-wide plane (N = 128, N1 = 8,
// N2 = 16, KC = 8), the same transform as pencil_pairs<kDst> with cheaper
// addressing.  Every slot a job's lane t touches is 8m + (t ^ c), c a
// compile-time constant and m either a constant or t, 2t or 15 - t; the row
// swizzle f() has period 8, so the byte offset is (a per-lane base for m) +
// H[c] + (8 slots) * (constant part of m), H[c] = offset of slot t ^ c: one
// add per distinct (base, c) where the generic path computes the slot and
// its swizzle per access.
template <typename T, int P, int JOBS, int NT, bool COLS, typename Lane = DstLane<T, 7>>
__device__ __forceinline__ void dst_pairs128(T* __restrict__ lds, const Lane& L, const T scale,
                                             const int tid) {
    using S = DstShape<7>;
    constexpr int N = 128, N1 = 8, N2 = 16, KC = 8;
    static_assert(S::N1 == N1 && S::N2 == N2 && S::KC == KC, "N = 128 shape");
    static_assert(JOBS * N1 == NT, "one job per thread");
    using Sw = RowSwizzle<N1>;
    constexpr int ES = (int)sizeof(T);
    constexpr int ROW8 = COLS ? 8 * P * ES : 8 * ES;   // bytes of 8 slots
    constexpr int PBO = COLS ? JOBS * ES : JOBS * P * ES;   // pencil g + JOBS (f(g + JOBS) = f(g))
    static_assert(JOBS % N1 == 0, "swizzle period");
    const int t = tid & (N1 - 1);
    const int g = tid / N1;
    char* const base = reinterpret_cast<char*>(lds);
    auto rowb = [&](int r) { return COLS ? (r * P + Sw::f(r)) * ES : r * ES; };   // slot r of pencil 0
    int H[N1];
#pragma unroll
    for (int c = 0; c < N1; ++c) H[c] = opaque(rowb(t ^ c));
    const int pb = COLS ? g * ES : (g * P + Sw::f(g)) * ES;
    const int b0 = opaque(pb), b1 = opaque(pb + ROW8 * t), b2 = opaque(pb + 2 * ROW8 * t),
              b3 = opaque(pb + ROW8 * (15 - t));
    // the slots outside the 8m + (t ^ c) form: N - t (step 1, j = t) and the
    // mirror of k = 8t (step 3)
    const int rA = opaque(pb + rowb((N - t) & (N - 1)));
    const int rB = opaque(pb + rowb(8 - t));   // f(8) = f(0): row 8(15 - j2) + 8 - t for every t
    const int rC = opaque(pb + rowb(S::posZ((N - 8 * t) & (N - 1))));
    // A ds instruction carries a byte offset below 64 KiB.  When 8 row groups
    // of the plane span more (FP64 columns), the accesses 8..15 row groups on
    // go from bases set 8 groups further (one add each, once per pass) instead
    // of an add per access.
    constexpr bool HI = COLS && 15 * ROW8 > 65535;
    const int b0h = HI ? opaque(pb + 8 * ROW8) : b0, rBh = HI ? opaque(rB + 8 * ROW8) : rB,
              b1h = HI ? opaque(b1 + 8 * ROW8) : b1;
    // lane base + c: c < 8 groups from `lo`, else from `hi` (8 groups on)
    auto split = [&](int lo, int hi, int lane, int groups) {
        return (HI && groups >= 8) ? hi + lane + ROW8 * (groups - 8) : lo + lane + ROW8 * groups;
    };
    auto A = [&](int off) -> T& { return *reinterpret_cast<T*>(base + off); };
    auto B = [&](int off) -> T& { return *reinterpret_cast<T*>(base + off + PBO); };

    // ---- step 1: pre-processing + 16-point DFTs over j2 (j = t + 8 j2)
    T yr[N2], yi[N2];
#pragma unroll
    for (int j2 = 0; j2 < N2; ++j2) {
        const int o0 = split(b0, b0h, H[0], j2);
        const int o1 = j2 == 0 ? rA : split(rB, rBh, 0, 15 - j2);
        const T a0 = A(o0), a1 = A(o1), c0 = B(o0), c1 = B(o1);
        const T sp = L.sine(j2);
        yr[j2] = fma(sp, a0 + a1, -a1);
        yi[j2] = fma(sp, c0 + c1, -c1);
    }
    dft<N2>(yr, yi);
#pragma unroll
    for (int k2 = 1; k2 < N2; ++k2) {
        T c, s;
        L.twiddle(k2, c, s);
        rotate(yr[k2], yi[k2], c, s);
    }
    wave_lds_sync();
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) {   // slot 8 k2 + (t ^ (k2 mod 8))
        const int o = b0 + H[k2 & 7] + ROW8 * k2;
        A(o) = yr[k2];
        B(o) = yi[k2];
    }
    wave_lds_sync();

    // ---- step 2: 8-point DFTs over j1 for k2 = t + 8 r (slot 8t + (j1 ^ t) + 64 r)
    T zr[N2], zi[N2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        T vr[N1], vi[N1];
#pragma unroll
        for (int j1 = 0; j1 < N1; ++j1) {
            const int o = split(b1, b1h, H[j1], 8 * r);
            vr[j1] = A(o);
            vi[j1] = B(o);
        }
        dft<N1>(vr, vi);
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) {
            zr[r * N1 + k1] = vr[k1];
            zi[r * N1 + k1] = vi[k1];
        }
    }
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) {   // posZ(t + cz) = cz + (t ^ ((r + 2 k1) mod 8)), cz = 8 (r + 2 k1)
            const int m = r + 2 * k1;
            const int o = split(b0, b0h, H[m & 7], m);
            A(o) = zr[r * N1 + k1];
            B(o) = zi[r * N1 + k1];
        }
    }
    wave_lds_sync();

    // ---- step 3: even outputs directly, odd outputs by prefix sum (as pencil_pairs)
    const T hs = T(0.5) * scale;
    T ae[KC], ao[KC], be[KC], bo[KC];
    T runA = T(0), runB = T(0);
#pragma unroll
    for (int i = 0; i < KC; ++i) {
        // posZ(8t + i) = 8t + (i ^ t); posZ(N - 8t - i) = 8 (15 - t) + (t ^ (7 ^ (8 - i))) for i > 0
        const int ok = b1 + H[i];
        const int on = i == 0 ? rC : b3 + H[7 ^ (8 - i)];
        const T zkr = A(ok), zki = B(ok);
        const T znr = A(on), zni = B(on);
        ae[i] = zni - zki;
        be[i] = zkr - znr;
        T dA = zkr + znr;
        T dB = zki + zni;
        if (i == 0 && t == 0) {
            dA *= T(0.5);
            dB *= T(0.5);
        }
        runA += dA;
        runB += dB;
        ao[i] = runA;
        bo[i] = runB;
    }
    const T offA = lane_scan_incl<N1>(runA) - runA;
    const T offB = lane_scan_incl<N1>(runB) - runB;
#pragma unroll
    for (int i = 0; i < KC; ++i) {
        ao[i] += offA;
        bo[i] += offB;
    }
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < KC; ++i) {
        // sigma(2k + e) for k = 8t + i: 16t + ((2i + e) mod 8 ^ t) + 8 ((2i + e) div 8)
        const bool k0 = i == 0 && t == 0;
        const int me = 2 * i, mo = 2 * i + 1;
        const int oe = b2 + H[me & 7] + ROW8 * (me >> 3), oo = b2 + H[mo & 7] + ROW8 * (mo >> 3);
        A(oe) = k0 ? T(0) : ae[i] * hs;
        B(oe) = k0 ? T(0) : be[i] * hs;
        A(oo) = ao[i] * hs;
        B(oo) = bo[i] * hs;
    }
    wave_lds_sync();
}

// ---------------------------------------------------------------------------
// The DST-I of N = 256 or 512 points with N/8 lanes to a pair of pencils.
//
// The packed FFT is 8 x 8 x R, R = N/64: L = N/8 lanes hold eight points each,
// so a lane's work between exchanges is one dft<8>.  (As 16 lanes of a 32-point
// and two 16-point DFTs, a pass of 511 x 511 FP64 points took 14.7 us: 32 blocks of
// two wavefronts, each a chain of some 1600 FP64 instructions with nothing
// beside it.)
//   j = t + L j2, t = p + R n;  k = k2 + 8 (m + 8 q), m = s + R e
//   1. DFT over j2 -> k2, times w_N^{t k2}       lane t -> lanes (k2, p)
//   2. DFT over n  -> m,  times w_L^{p m}        lane (k2, p) -> (k2, s)
//   3. DFT over p  -> q                          Z_k, then step 3 of pencil_pairs
// Exchanges go through the pencils' own slots.  The swizzles are linear over the
// bits of the index, chosen so that 32 consecutive lanes read and 16 write
// distinct banks of eight bytes:
//   exchange 1:  slot L k2 + (t ^ x),                 x = R k2 mod 32
//   exchange 2:  slot L k2 + ((8 p + (m ^ p)) ^ x)
//   Z:           posZ: bits 4, 5, 6 of k into bits 2, 1, 0
//   outputs:     sigma: bits 4, 5, 6 of j into bits 0, 1, 2
// ---------------------------------------------------------------------------
template <typename T, int LOGN>
struct WaveDst {
    static constexpr int N = 1 << LOGN, L = N / 8, R = L / 8, E = 8 / R;
    static_assert(L == 32 || L == 64, "half or all of a wavefront");
    T twr[8], twi[8];   // w_N^{t k}
    T ur[8], ui[8];     // w_L^{(t mod R) m}
    T sp[8];            // sin(pi (t + L j)/N) + 1/2
    __device__ static constexpr int posZ(int k) {
        return k ^ ((k >> 6) & 1) ^ (((k >> 5) & 1) << 1) ^ (((k >> 4) & 1) << 2);
    }
    __device__ static constexpr int sigma(int j) { return j ^ ((j >> 4) & 7); }
    // slot of output point m (as PencilIO<kDst>::out)
    __device__ static constexpr int out(int m) { return sigma(m + 1); }
    // tables as DstLane::init
    __device__ __forceinline__ void init(const T* __restrict__ tables, const int t) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            sp[k] = tables[2 * N + t + L * k];
            if (k == 0) continue;
            twr[k] = tables[t * k];
            twi[k] = tables[N + t * k];
            ur[k] = tables[8 * (t % R) * k];
            ui[k] = tables[N + 8 * (t % R) * k];
        }
    }

    // The pencils a and b (N slots each, points in natural order from slot 1,
    // slot 0 finite), transformed in place by the L lanes t.
    __device__ __forceinline__ void pair(T* __restrict__ a, T* __restrict__ b, const T scale, const int t) const {
        T yr[8], yi[8];
        const int m0 = (N - t) & (N - 1);
#pragma unroll
        for (int j = 0; j < 8; ++j) {   // N - (t + L j) = L - t + L (7 - j) but for t = j = 0
            const int o = t + L * j, n = j == 0 ? m0 : L - t + L * (7 - j);
            const T a0 = a[o], a1 = a[n], b0 = b[o], b1 = b[n];
            yr[j] = fma(sp[j], a0 + a1, -a1);
            yi[j] = fma(sp[j], b0 + b1, -b1);
        }
        dft<8>(yr, yi);
#pragma unroll
        for (int k = 1; k < 8; ++k) rotate(yr[k], yi[k], twr[k], twi[k]);
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int o = L * k + (t ^ (R * k & 31));
            a[o] = yr[k];
            b[o] = yi[k];
        }
        wave_lds_sync();
        const int k2 = t / R, p = t % R, x = R * k2 & 31;
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const int o = L * k2 + p + ((R * n & 31) ^ x) + (R * n & 32);
            yr[n] = a[o];
            yi[n] = b[o];
        }
        dft<8>(yr, yi);
#pragma unroll
        for (int m = 1; m < 8; ++m) rotate(yr[m], yi[m], ur[m], ui[m]);
        wave_lds_sync();
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int o = L * k2 + ((8 * p + (m ^ p)) ^ x);
            a[o] = yr[m];
            b[o] = yi[m];
        }
        wave_lds_sync();
#pragma unroll
        for (int e = 0; e < E; ++e) {   // lane (k2, s = p)
            T vr[R], vi[R];
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int o = L * k2 + ((8 * q + ((p + R * e) ^ q)) ^ x);
                vr[q] = a[o];
                vi[q] = b[o];
            }
            dft<R>(vr, vi);
#pragma unroll
            for (int q = 0; q < R; ++q) {
                yr[R * e + q] = vr[q];
                yi[R * e + q] = vi[q];
            }
        }
        wave_lds_sync();
        const int z = posZ(k2 + 8 * p);
#pragma unroll
        for (int e = 0; e < E; ++e) {
#pragma unroll
            for (int q = 0; q < R; ++q) {   // posZ of the constant part: its own bits, and 5 and 6 into 1 and 0
                const int c = 8 * R * e + 64 * q, o = (z ^ (posZ(c) ^ c)) + c;
                a[o] = yr[R * e + q];
                b[o] = yi[R * e + q];
            }
        }
        wave_lds_sync();
        // even outputs directly, odd ones by prefix sum; lane t owns k = 4 t + i
        const T hs = T(0.5) * scale;
        T ae[4], ao[4], be[4], bo[4];
        T runA = T(0), runB = T(0);
        const int zk = posZ(4 * t), z0 = posZ((N - 4 * t) & (N - 1)), zn = posZ(4 * (2 * L - 1 - t));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = zk ^ i, n = i == 0 ? z0 : zn ^ (4 - i);
            const T zkr = a[k], zki = b[k], znr = a[n], zni = b[n];
            ae[i] = zni - zki;
            be[i] = zkr - znr;
            T dA = zkr + znr, dB = zki + zni;
            if (i == 0 && t == 0) {
                dA *= T(0.5);
                dB *= T(0.5);
            }
            runA += dA;
            runB += dB;
            ao[i] = runA;
            bo[i] = runB;
        }
        const T offA = wave_scan_incl<L>(runA) - runA, offB = wave_scan_incl<L>(runB) - runB;
        wave_lds_sync();
        const int sw = (t >> 1) & 7;
#pragma unroll
        for (int i = 0; i < 4; ++i) {   // sigma(8 t + c) = 8 t + (c ^ sw)
            const bool k0 = i == 0 && t == 0;
            const int e = 8 * t + ((2 * i) ^ sw), o = 8 * t + ((2 * i + 1) ^ sw);
            a[e] = k0 ? T(0) : ae[i] * hs;
            b[e] = k0 ? T(0) : be[i] * hs;
            a[o] = (ao[i] + offA) * hs;
            b[o] = (bo[i] + offB) * hs;
        }
        wave_lds_sync();
    }
};

// ---------------------------------------------------------------------------
// pencil_pairs<KIND> for all rows (COLS false) or columns (COLS true) of a 128 x
// 128 plane, 16 lanes of eight points to a pair of pencils: 1024 threads, one job
// each.
//
// The packed FFT is 8 x 8 x 2 (WaveDst with L = 16, R = 2); the radix-2 stage
// stays in registers, its operands exchanged with the neighbouring lane by DPP,
// so a pass makes the four trips through LDS that pencil_pairs makes with 8
// lanes of 16 points, with half the registers a thread and twice the wavefronts
// to hide their latency.
//
// Layout: rows of pitch P = 129, no swizzle; a job takes pencils q and q + 1, the
// two jobs of 32 lanes pencils 16 apart.  In every access a job's 16 lanes take
// slots distinct mod 16, and 16 rows or columns are 16 banks mod 32: by banks of
// eight bytes no read of 32 lanes or write of 16 meets a conflict.  The counters
// show 0.25 conflict cycles an LDS instruction in the streaming kernel, staging and
// store phase included, where the 8-lane form's skewed layout had 0.14: what the
// form gains it gains by the wavefronts.
// Slots: exchange 1 at 16 k2 + (t ^ 2 k2); Z by posZ (bits 4, 5 of k into bits
// 0, 1, bit 6 into bit 3), where the periodic kinds leave their outputs; DST
// outputs by sigma, as DstShape<7>.
// ---------------------------------------------------------------------------
constexpr int kWidePitch = 129;
__device__ constexpr int wide_posZ(int k) { return k ^ ((k >> 4) & 3) ^ (((k >> 6) & 1) << 3); }
// slot that holds output point m (as PencilIO::out)
template <int KIND>
__device__ constexpr int wide_out(int m) {
    return KIND == kDst ? DstShape<7>::sigma(m + 1) : wide_posZ(m);
}

// Lane t's constants in LDS (held in registers they would spill what a streaming
// kernel prefetches): the shifted sines, then w_128^{t k} as [k - 1][t] pairs.
template <typename T>
struct Wide128Lane {
    static constexpr int kValues = 128 + 2 * 16 * 7;
    const T* sl;
    const T* tl;
    __device__ static void fill(const T* __restrict__ tables, T* lds, const int tid, const int nt) {
        for (int m = tid; m < 128; m += nt) lds[m] = tables[256 + m];
        for (int m = tid; m < 16 * 7; m += nt) {
            const int tk = (m & 15) * (m / 16 + 1);
            lds[128 + 2 * m] = tables[tk];
            lds[128 + 2 * m + 1] = tables[128 + tk];
        }
    }
    __device__ __forceinline__ Wide128Lane(const T* lds, const int t) : sl(lds + t), tl(lds + 128 + 2 * t) {}
};

template <int KIND, bool COLS, typename T>
__device__ __forceinline__ void wide_pairs128(T* __restrict__ lds, const Wide128Lane<T>& L, const T scale,
                                              const int tid) {
    constexpr int N = 128, P = kWidePitch, ES = (int)sizeof(T);
    constexpr int SB = (COLS ? P : 1) * ES, DB = (COLS ? 1 : P) * ES;   // bytes from slot to slot, pencil to pencil
    constexpr bool HI = 127 * SB + DB > 65535;   // more than a ds instruction's offset carries
    const int t = tid & 15, p = t & 1, k2 = t >> 1, g = tid >> 4;
    const int q = 32 * (g >> 4) + 2 * ((g >> 1) & 7) + 16 * (g & 1);
    const int pb = opaque(q * DB), ph = HI ? opaque(pb + 64 * SB) : pb;
    char* const mem = reinterpret_cast<char*>(lds);
    // slot `lane` + c of pencil q, c a compile-time constant
    auto at = [&](const int lane, const int c) -> T* {
        return reinterpret_cast<T*>(mem + (HI && c >= 64 ? ph + lane * SB + (c - 64) * SB : pb + lane * SB + c * SB));
    };
    auto B = [](T* a) -> T& { return *reinterpret_cast<T*>(reinterpret_cast<char*>(a) + DB); };

    T yr[8], yi[8];
    const int m0 = (N - t) & (N - 1);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        T* a = at(t, 16 * j);
        const T a0 = *a, b0 = B(a);
        if constexpr (KIND == kRdftFwd) {
            yr[j] = a0;
            yi[j] = b0;
        } else {
            T* n = j == 0 ? at(m0, 0) : at(16 - t, 16 * (7 - j));
            const T a1 = *n, b1 = B(n);
            if constexpr (KIND == kDst) {
                const T sp = L.sl[16 * j];
                yr[j] = fma(sp, a0 + a1, -a1);
                yi[j] = fma(sp, b0 + b1, -b1);
            } else {   // points t + 16 j below N/2, then above; 0 and N/2 stand alone
                const bool edge = (j == 0 || j == 4) && t == 0;
                yr[j] = edge ? T(0.5) * a0 : j < 4 ? T(0.5) * (a0 + b1) : T(0.5) * (a1 - b0);
                yi[j] = edge ? T(-0.5) * b0 : j < 4 ? T(0.5) * (a1 - b0) : T(-0.5) * (a0 + b1);
            }
        }
    }
    dft<8>(yr, yi);
#pragma unroll
    for (int k = 1; k < 8; ++k) rotate(yr[k], yi[k], L.tl[32 * (k - 1)], L.tl[32 * (k - 1) + 1]);
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        T* a = at(t ^ (2 * k), 16 * k);
        *a = yr[k];
        B(a) = yi[k];
    }
    wave_lds_sync();
#pragma unroll
    for (int n = 0; n < 8; ++n) {
        T* a = at(16 * k2 + p + 2 * (n ^ k2), 0);
        yr[n] = *a;
        yi[n] = B(a);
    }
    dft<8>(yr, yi);
    // lane p: the odd points' twiddles w_16^m, then self + other (p = 0) or other - self
    const T sg = p ? T(-1) : T(1);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        if (m > 0) rotate(yr[m], yi[m], p ? (T)cos32(2 * m) : T(1), p ? (T)-sin32(2 * m) : T(0));
        yr[m] = fma(sg, yr[m], lane_xor1(yr[m]));
        yi[m] = fma(sg, yi[m], lane_xor1(yi[m]));
    }
    wave_lds_sync();
    const int z = k2 + 8 * p;
#pragma unroll
    for (int m = 0; m < 8; ++m) {   // k = k2 + 8 m + 64 p
        T* a = at((z ^ ((m >> 1) + 8 * (m & 1))) + 64 * p, 16 * (m >> 1));
        *a = KIND == kRdftInv ? yr[m] * scale : yr[m];      // x^a = Re Y, x^b = -Im Y
        B(a) = KIND == kRdftInv ? -yi[m] * scale : yi[m];
    }
    wave_lds_sync();
    if constexpr (KIND == kRdftInv) return;
    const int zk = wide_posZ(4 * t), z0 = wide_posZ((N - 4 * t) & (N - 1)), zn = wide_posZ(4 * (31 - t));
    if constexpr (KIND == kRdftFwd) {
        // split the packed spectra: lane t owns k = 4 t + i and the mirrors N - k
        // (k = 0: the Nyquist slot N/2)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool k0 = i == 0 && t == 0;
            T *k = at(zk ^ i, 0), *n = at(i == 0 ? (t == 0 ? wide_posZ(N / 2) : z0) : zn ^ (4 - i), 0);
            const T zkr = *k, zki = B(k), znr = *n, zni = B(n);
            *k = (k0 ? zkr : T(0.5) * (zkr + znr)) * scale;
            B(k) = (k0 ? zki : T(0.5) * (zki + zni)) * scale;
            *n = (k0 ? znr : T(0.5) * (zni - zki)) * scale;
            B(n) = (k0 ? zni : T(0.5) * (zkr - znr)) * scale;
        }
        wave_lds_sync();
        return;
    }
    // even outputs directly, odd ones by prefix sum; lane t owns k = 4 t + i
    const T hs = T(0.5) * scale;
    T ae[4], ao[4], be[4], bo[4];
    T runA = T(0), runB = T(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        T *k = at(zk ^ i, 0), *n = at(i == 0 ? z0 : zn ^ (4 - i), 0);
        const T zkr = *k, zki = B(k), znr = *n, zni = B(n);
        ae[i] = zni - zki;
        be[i] = zkr - znr;
        T dA = zkr + znr, dB = zki + zni;
        if (i == 0 && t == 0) {
            dA *= T(0.5);
            dB *= T(0.5);
        }
        runA += dA;
        runB += dB;
        ao[i] = runA;
        bo[i] = runB;
    }
    const T offA = wave_scan_incl<16>(runA) - runA, offB = wave_scan_incl<16>(runB) - runB;
    wave_lds_sync();
    const int sw = (t >> 1) & 7;
#pragma unroll
    for (int i = 0; i < 4; ++i) {   // sigma(8 t + c) = 8 t + (c ^ sw)
        const bool k0 = i == 0 && t == 0;
        T *e = at(8 * t + ((2 * i) ^ sw), 0), *o = at(8 * t + ((2 * i + 1) ^ sw), 0);
        *e = k0 ? T(0) : ae[i] * hs;
        B(e) = k0 ? T(0) : be[i] * hs;
        *o = (ao[i] + offA) * hs;
        B(o) = (bo[i] + offB) * hs;
    }
    wave_lds_sync();
}

// ---------------------------------------------------------------------------
// Constant-coefficient cyclic reduction along z for one (kx,ky) mode.
//
// After the DST in x and y, mode (kx,ky) obeys the Toeplitz tridiagonal system
//   b u_{i-1} + d u_i + b u_{i+1} = g_i,  i = 0..n-1,  n = 2^Q - 1,
//   b = 1/hz^2, d = -2/hz^2 - lambda_x[kx] - lambda_y[ky], u_{-1} = u_n = 0,
// the system the reference's z DST + divide + inverse z DST solves
// (src/lapl_cube.cpp:13-30, 70-80, 124-141).  Odd-even cyclic reduction
// (Hockney & Jesshope, the reference's cyclic_reduction,
// src/cyclic_reduction.h:20-56) keeps the coefficients uniform at every level
// when n = 2^Q - 1, so each level is two scalars per mode:
//   alpha_l = -c_{l-1}/d_{l-1},  d_l = d_{l-1} - 2 c_{l-1}^2/d_{l-1},
//   c_l = -c_{l-1}^2/d_{l-1}.
// The diagonal is carried as its excess s = -d - 2 c over the couplings (s_0 =
// lambda_x + lambda_y), which a level multiplies by 1 + 2 alpha: every quantity
// is a sum or product of positive terms, so the lowest modes' systems, where d
// and 2 c nearly cancel, keep full relative accuracy.  (Carried as d, FP32
// elimination loses 1e-4 of those modes at 128 rows, FP64 1e-13.)
// G lanes share one system: lane c owns the contiguous chunk of rows
// [c*C, (c+1)*C - 1) plus the separator row (c+1)*C - 1 (C = 2^Q/G).  The
// lowest Q-g levels stay inside a chunk; the separators' updates are additive
// so each lane accumulates its contribution to its two neighbouring
// separators and one shuffle combines them; the remaining g-1 levels over the
// G-1 separators are solved redundantly in every lane from shuffled values.
// ---------------------------------------------------------------------------
template <typename T, int Q>
struct CrLevels {
    T alpha[Q > 1 ? Q : 2];   // alpha[l], l = 1..Q-1
    T c[Q];                   // c[l],  l = 0..Q-1
    T inv_d[Q];               // 1/d[l], l = 0..Q-1
};

// One level's scalars from (c, s), and the next level's (c, s).
template <typename T>
__device__ __forceinline__ void cr_level(T& c, T& s, T& inv_d, T& alpha) {
    const T inv = T(1) / fma(T(2), c, s);   // -1/d
    inv_d = -inv;
    alpha = c * inv;
    c *= alpha;
    s = fma(T(2) * alpha, s, s);
}

// c = b, s = lambda_x + lambda_y
template <typename T, int Q>
__device__ __forceinline__ void cr_levels(CrLevels<T, Q>& L, T c, T s) {
#pragma unroll
    for (int l = 0; l < Q; ++l) {
        L.c[l] = c;
        T a;
        cr_level(c, s, L.inv_d[l], a);
        if (l + 1 < Q) L.alpha[l + 1] = a;
    }
}

}  // namespace fdmgpu
