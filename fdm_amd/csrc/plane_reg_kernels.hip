// FP32 planes of N = 256 (gfx950): transforms along x and y of whole z-planes
// that do not fit LDS, held in registers between the two passes.
//
// A 256 x 256 plane of floats is 256 KB: more than a CU's 160 KB of LDS, half
// of its 512 KB of registers.  The axis tiles move such a plane through HBM
// once per axis; here one block of 1024 threads (16 waves, 128 registers each)
// owns the plane and moves it once.  LDS holds half of it at a time:
//   first pass:  128 rows at a time (pencils = rows), the outputs into 32
//                registers per thread and half;
//   second pass: 128 columns at a time (pencils = columns, all 256 rows), from
//                the registers, the outputs to global memory
// (the inverse: columns first, then rows).  The second half's rows are loaded while the first half is transformed (FP32
// input: all of them, FP64 input: half, the registers allow no more), and the
// first half's stores drain while the second half is transformed.
//
// Answers are bitwise those of the axis tiles at their default sizes (x tiles
// of 32 rows of one plane, y tiles of 64 columns): the axes go in the tiles'
// order, and, as two pencils share a complex transform and a pencil's rounding
// depends on its partner, the partners are the tiles': rows y and y + 16 of 32,
// columns x and x + 32 of 64.  Which of the two runs may therefore depend on the
// batch.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "dst_device.hpp"
#include "kernel_util.hpp"
#include "kernels.hpp"

namespace fdmgpu {

// LDS layout of a half: pencil-major, PITCH slots a pencil, slot j of pencil q
// at q PITCH + (j ^ h(q)).  PITCH is 16 mod 32 banks and a multiple of 16, so
//  * a pass is conflict-free: the two jobs of 16 lanes in a half-wavefront take
//    neighbouring pencils, in the two halves of the 32 banks;
//  * every slot a pass touches is 16 m + (t ^ c) with c a compile-time constant,
//    so its byte address is one exclusive-or of a lane base with 4 c, plus an
//    offset the ds instruction carries.  With the additive row shift of the
//    other plane kernels a wave issued 4200 VALU instructions instead of 3050
//    and 1009 LDS instructions instead of 789: 51 us a launch of 255 FP32
//    planes, 46 with this layout.
// Rows (ROWS) go in and out along their slots: h = 0.  Columns are written and
// read 32 neighbouring pencils at a time: h(q) = (q / 2) mod 16 spreads them over
// all banks.
constexpr int kHalfPitch = 272, kHalfPB = kHalfPitch * 4;   // slots, bytes a pencil
template <bool ROWS>
struct HalfLayout {
    static constexpr int DP = ROWS ? 16 : 32;   // a job's pencils: q and q + DP of 2 DP
    __device__ static constexpr int h(int q) { return ROWS ? 0 : (q >> 1) & 15; }
    __device__ static constexpr int pencil(int job) { return (job & (DP - 1)) + (job / DP) * 2 * DP; }
    __device__ static constexpr int byte(int q, int j) { return q * kHalfPB + ((j ^ h(q)) << 2); }
};

struct PlaneRegCfg {
    static constexpr int LOGN = 8, N = 256, NT = 1024, HALF = 128;
    using S = DstShape<LOGN>;
    static constexpr int SLOTS = HALF * kHalfPitch;
    using Lane = DstLaneLds<float, LOGN>;
    static constexpr size_t lds_bytes() { return sizeof(float) * (size_t)(SLOTS + Lane::kValues); }
    static_assert(S::N1 == 16 && S::N2 == 16 && S::KC == 8, "N = 256 shape");
    // slot of FFT output Z_k: posZ with one more term, so that step 3's 32
    // lanes (k = 8 t + i, two jobs) hit 32 banks (posZ: 16, 9% of the LDS cycles)
    __device__ static constexpr int pz(int k) { return (k & ~7) | ((k ^ (k >> 3) ^ (k >> 6)) & 7); }
    // slot of output j (kDst: point j - 1)
    __device__ static constexpr int out(int kind, int j) { return kind == kDst ? S::sigma(j) : pz(j); }
    static_assert((HALF / 2) * S::N1 == NT, "one job lane per thread");
};

// pencil_pairs<KIND> of dst_device.hpp for the 128 pencils of a half: the same
// transform, operation for operation.
template <int KIND, bool ROWS>
__device__ __forceinline__ void half_pencils(float* __restrict__ lds, const PlaneRegCfg::Lane& L, const float scale,
                                             const int tid) {
    using C = PlaneRegCfg;
    constexpr int N = C::N, N2 = C::S::N2, KC = C::S::KC;
    using Lay = HalfLayout<ROWS>;
    constexpr int DB = Lay::DP * kHalfPB;
    static_assert(Lay::h(5) == Lay::h(5 + Lay::DP), "a job's pencils share h");
    const int t = tid & 15, q = Lay::pencil(tid >> 4);
    const int h = Lay::h(q), pb = q * kHalfPB;
    char* const mem = reinterpret_cast<char*>(lds);
    auto A = [&](int off) -> float& { return *reinterpret_cast<float*>(mem + off); };
    auto B = [&](int off) -> float& { return *reinterpret_cast<float*>(mem + off + DB); };
    auto slot = [&](int j) { return pb + ((j ^ h) << 2); };   // any slot, computed
    const int b0 = opaque(slot(t)), b1 = opaque(b0 + (t << 6));

    // ---- step 1 (slots t + 16 j2 and their mirrors N - j)
    float yr[N2], yi[N2];
    {
        const int rA = opaque(slot((N - t) & (N - 1))), rB = opaque(t ? slot(16 - t) : 64 + slot(0));
#pragma unroll
        for (int j2 = 0; j2 < N2; ++j2) {
            const int j = t + 16 * j2, o0 = b0 + 64 * j2, o1 = j2 == 0 ? rA : rB + 64 * (15 - j2);
            if constexpr (KIND == kRdftFwd) {
                yr[j2] = A(o0);
                yi[j2] = B(o0);
            } else {
                const float a0 = A(o0), a1 = A(o1), c0 = B(o0), c1 = B(o1);
                if constexpr (KIND == kDst) {
                    const float sp = L.sine(j2);
                    yr[j2] = fma(sp, a0 + a1, -a1);
                    yi[j2] = fma(sp, c0 + c1, -c1);
                } else if (2 * j2 < N2) {
                    const bool edge = j == 0;
                    yr[j2] = edge ? 0.5f * a0 : 0.5f * (a0 + c1);
                    yi[j2] = edge ? -0.5f * c0 : 0.5f * (a1 - c0);
                } else {
                    const bool edge = j == N / 2;
                    yr[j2] = edge ? 0.5f * a0 : 0.5f * (a1 - c0);
                    yi[j2] = edge ? -0.5f * c0 : -0.5f * (a0 + c1);
                }
            }
        }
    }
    dft<N2>(yr, yi);
#pragma unroll
    for (int k2 = 1; k2 < N2; ++k2) {
        float c, s;
        L.twiddle(k2, c, s);
        rotate(yr[k2], yi[k2], c, s);
    }
    wave_lds_sync();
#pragma unroll
    for (int k2 = 0; k2 < N2; ++k2) {   // slot 16 k2 + (t ^ k2)
        const int o = (b0 ^ (4 * k2)) + 64 * k2;
        A(o) = yr[k2];
        B(o) = yi[k2];
    }
    wave_lds_sync();

    // ---- step 2: 16-point DFTs over j1 for k2 = t (slot 16 t + (j1 ^ t))
    float zr[16], zi[16];
#pragma unroll
    for (int j1 = 0; j1 < 16; ++j1) {
        const int o = b1 ^ (4 * j1);
        zr[j1] = A(o);
        zi[j1] = B(o);
    }
    dft<16>(zr, zi);
    wave_lds_sync();
    {
        // k = t + 16 k1: pz(k) = 16 k1 + (t ^ t / 8 ^ 2 k1 mod 8 ^ k1 / 4)
        const int bz = opaque(slot(t ^ (t >> 3)));
#pragma unroll
        for (int k1 = 0; k1 < 16; ++k1) {
            const int o = (bz ^ (4 * (((2 * k1) & 7) ^ (k1 >> 2)))) + 64 * k1;
            if constexpr (KIND == kRdftInv) {
                A(o) = zr[k1] * scale;
                B(o) = -zi[k1] * scale;
            } else {
                A(o) = zr[k1];
                B(o) = zi[k1];
            }
        }
    }
    wave_lds_sync();

    if constexpr (KIND != kRdftInv) {
        // ---- step 3: lane t owns k = 8 t + i and their mirrors N - k:
        // slots pz(8 t) ^ i, and for i > 0 the mirrors pz(8 (31 - t)) ^ (8 - i)
        const int b2 = opaque(slot(C::pz(8 * t))), b3 = opaque(slot(C::pz(8 * (31 - t))));
        auto ok = [&](int i) { return b2 ^ (4 * i); };
        if constexpr (KIND == kRdftFwd) {
            const int rC = opaque(slot(C::pz(t == 0 ? N / 2 : N - 8 * t)));
#pragma unroll
            for (int i = 0; i < KC; ++i) {
                const bool k0 = i == 0 && t == 0;
                const int pk = ok(i), pn = i == 0 ? rC : b3 ^ (4 * (8 - i));
                const float zkr = A(pk), zki = B(pk), znr = A(pn), zni = B(pn);
                A(pk) = (k0 ? zkr : 0.5f * (zkr + znr)) * scale;
                B(pk) = (k0 ? zki : 0.5f * (zki + zni)) * scale;
                A(pn) = (k0 ? znr : 0.5f * (zni - zki)) * scale;
                B(pn) = (k0 ? zni : 0.5f * (zkr - znr)) * scale;
            }
        } else {
            const int rC = opaque(slot(C::pz((N - 8 * t) & (N - 1))));
            const float hs = 0.5f * scale;
            float ae[KC], ao[KC], be[KC], bo[KC];
            float runA = 0.f, runB = 0.f;
#pragma unroll
            for (int i = 0; i < KC; ++i) {
                const int pk = ok(i), pn = i == 0 ? rC : b3 ^ (4 * (8 - i));
                const float zkr = A(pk), zki = B(pk), znr = A(pn), zni = B(pn);
                ae[i] = zni - zki;
                be[i] = zkr - znr;
                float dA = zkr + znr, dB = zki + zni;
                if (i == 0 && t == 0) {
                    dA *= 0.5f;
                    dB *= 0.5f;
                }
                runA += dA;
                runB += dB;
                ao[i] = runA;
                bo[i] = runB;
            }
            const float offA = lane_scan_incl<16>(runA) - runA;
            const float offB = lane_scan_incl<16>(runB) - runB;
            wave_lds_sync();
#pragma unroll
            for (int i = 0; i < KC; ++i) {   // sigma(16 t + 2 i + e) = 16 t + ((2 i + e) ^ t)
                const bool k0 = i == 0 && t == 0;
                const int oe = b1 ^ (4 * (2 * i)), oo = b1 ^ (4 * (2 * i + 1));
                A(oe) = k0 ? 0.f : ae[i] * hs;
                B(oe) = k0 ? 0.f : be[i] * hs;
                A(oo) = (ao[i] + offA) * hs;
                B(oo) = (bo[i] + offB) * hs;
            }
        }
        wave_lds_sync();
    }
}

// ACC and KIND as plane_dst_kernel's.  INV: columns first, then rows (the order
// of the axis tiles' inverse); else rows first.
template <typename Tin, typename Tout, int ACC, int KIND, bool INV>
__global__ __launch_bounds__(PlaneRegCfg::NT) __attribute__((amdgpu_waves_per_eu(4))) void plane_reg_kernel(
    const BatchPtr<const Tin> in, const BatchPtr<Tout> out, const float s1, const float s2,
    const float* __restrict__ tables, const int* __restrict__ done, const float* __restrict__ base,
    const long base_bs, int* __restrict__ reset) {
    using C = PlaneRegCfg;
    using IO = PencilIO<KIND, C::LOGN>;
    using LR = HalfLayout<true>;    // rows
    using LC = HalfLayout<false>;   // columns
    constexpr int N = C::N, NT = C::NT, HALF = C::HALF, PB = kHalfPB;
    constexpr int n = IO::n, o = IO::off;
    const int tid = threadIdx.x, p = blockIdx.y;
    const long plane_off = (long)blockIdx.x * n * n;
    constexpr unsigned pts = (unsigned)n * n;
    const BufRange<Tout> dst(wave_uniform(out.uniform(p)) + plane_off, pts * sizeof(Tout));
    [[maybe_unused]] const BufRange<float> bp(ACC == 2 ? base + p * base_bs + plane_off : (const float*)nullptr,
                                              ACC == 2 ? pts * (unsigned)sizeof(float) : 0u);
    // A thread index the compiler cannot carry through a pass: addresses are
    // formed where they are used (kept live through the passes they spill).
    auto fresh = [&] {
        int t = tid;
        asm volatile("" : "+v"(t));
        return t;
    };
    // Two thread maps, each 32 elements a thread and half plane.  By rows:
    // column x = tid mod 256 of rows r0 + 4 i of 128; by columns: column s = tid
    // mod 128 of rows q0 + 8 i of 256.  Elements outside the plane address past
    // the buffer's range (loads read 0, stores are dropped): column 255 by an
    // offset of its own, row 255 by where it lies.
    constexpr int RR = NT / N, CR = NT / HALF, II = 32;
    const int r0 = __builtin_amdgcn_readfirstlane(tid / N), q0 = __builtin_amdgcn_readfirstlane(tid / HALF);
    auto row_lane = [&](const int x, const int es) { return x < n ? (r0 * n + x) * es : (int)pts * es; };
    auto row_so = [](const int half, const int i, const int es) { return (HALF * half + RR * i) * n * es; };
    auto col_lane = [&](const int x, const int es) { return x < n ? (q0 * n + x) * es : (int)pts * es; };
    if (done && done[p]) {
        if constexpr (ACC == 2) {
            const int x = tid & (N - 1);
            for (int half = 0; half < 2; ++half)
#pragma unroll 8
                for (int i = 0; i < II; ++i)
                    dst.store((Tout)bp.load(row_lane(x, 4), row_so(half, i, 4)), row_lane(x, sizeof(Tout)),
                              row_so(half, i, sizeof(Tout)));
        }
        return;
    }
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float* lds = reinterpret_cast<float*>(smem_raw);
    char* const mem = reinterpret_cast<char*>(smem_raw);
    auto at = [&](int off) -> float& { return *reinterpret_cast<float*>(mem + off); };
    const BufRange<Tin> src(wave_uniform(in.uniform(p)) + plane_off, pts * sizeof(Tin));

    using Lane = C::Lane;
    float* consts = lds + C::SLOTS;
    Lane L;
    Lane::fill(tables, consts, tid, NT);
    L.init(consts, tid & 15);

    // ---- first pass: half f of the rows (INV: of the columns)
    const int lane_in = INV ? 0 : row_lane(tid & (N - 1), sizeof(Tin));
    auto load = [&](const int f, const int i) {
        if constexpr (INV)
            return src.load(col_lane((tid & (HALF - 1)) + HALF * f, sizeof(Tin)), CR * i * n * (int)sizeof(Tin));
        else
            return src.load(lane_in, row_so(f, i, sizeof(Tin)));
    };
    // columns in LDS from v(i), row q0 + 8 i: row 255 (Dirichlet) falls on slot
    // 256, in the pad, and slot 0 is 0
    auto put_columns = [&](auto&& v) {
        const int s = fresh() & (HALF - 1);
        const int b[2] = {opaque(LC::byte(s, q0 + o)), opaque(LC::byte(s, q0 + 8 + o))};
#pragma unroll
        for (int i = 0; i < II; ++i) at(b[i & 1] + 64 * (i >> 1)) = v(i);
        if (KIND == kDst && q0 == CR - 1) at(LC::byte(s, 0)) = 0.f;
    };
    // slot 0 of the rows (a pass leaves it 0)
    auto zero_rows = [&] {
        if constexpr (KIND == kDst)
            for (int r = tid; r < HALF; r += NT) at(LR::byte(r, 0)) = 0.f;
    };
    Tin v[II];
    auto stage = [&] {
        if constexpr (INV) {
            put_columns([&](int i) { return (float)v[i]; });
        } else {
            const int b = opaque(LR::byte(r0, (fresh() & (N - 1)) + o));   // column 255: the pad
#pragma unroll
            for (int i = 0; i < II; ++i) at(b + RR * i * PB) = (float)v[i];
        }
    };
    // its outputs: w[f][c][i]
    //   rows first: column s + 128 c of row 128 f + q0 + 8 i, i < 16 (column 255:
    //               slot 0, which holds 0)
    //   columns first: column s + 128 f of row 128 c + q0 + 8 i (row 255: slot 0)
    constexpr int XI = HALF / CR;   // 16
    float w[2][2][XI];
    auto take = [&](const int f) {
        const int s = fresh() & (HALF - 1);
        if constexpr (INV) {
            const int b = opaque(LC::byte(s, 0));
#pragma unroll
            for (int i = 0; i < II; ++i) {
                const int y = q0 + CR * i, sl = y < n ? C::out(KIND, y + o) : 0;   // wave-uniform
                w[f][i / XI][i % XI] = at((b ^ (4 * (sl & 15))) + 64 * (sl >> 4));
            }
        } else {
            int b[2];
#pragma unroll
            for (int c = 0; c < 2; ++c)
                b[c] = opaque(LR::byte(q0, s + HALF * c < n ? C::out(KIND, s + HALF * c + o) : 0));
#pragma unroll
            for (int i = 0; i < XI; ++i)
#pragma unroll
                for (int c = 0; c < 2; ++c) w[f][c][i] = at(b[c] + CR * i * PB);
        }
    };
    constexpr int PF = sizeof(Tin) == 4 ? II : II / 2;   // of the second half, loaded during the first half's pass
#pragma unroll
    for (int i = 0; i < II; ++i) v[i] = load(0, i);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!INV) zero_rows();
    stage();
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PF; ++i) v[i] = load(1, i);
    __builtin_amdgcn_sched_barrier(0);
    half_pencils<KIND, !INV>(lds, L, s1, fresh());
    __syncthreads();
#pragma unroll
    for (int i = PF; i < II; ++i) v[i] = load(1, i);
    take(0);
    __syncthreads();
    stage();
    __syncthreads();
    half_pencils<KIND, !INV>(lds, L, s1, fresh());
    __syncthreads();
    take(1);
    __syncthreads();

    // ---- second pass and store: half f of the columns (INV: of the rows)
    if constexpr (INV) zero_rows();
    static_for<0, 2>([&](auto ff) {
        constexpr int f = decltype(ff)::value;
        if constexpr (INV) {
            const int s = fresh() & (HALF - 1);
            const int b = opaque(LR::byte(q0, s + o));
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int i = 0; i < XI; ++i) at(b + 4 * HALF * c + CR * i * PB) = w[c][f][i];
        } else {
            put_columns([&](int i) { return w[i / XI][f][i % XI]; });
        }
        __syncthreads();
        half_pencils<KIND, INV>(lds, L, s2, fresh());
        __syncthreads();
        // element i of the thread's 32: its LDS byte, and its global lane and
        // constant offsets for elements of es bytes.  Columns: output j = q0 + 8 i
        // (row j - o) sits in slot out(j): for the DST sigma(j) = 16 (i / 2) + (q0 ^
        // 8 (i mod 2) ^ i / 2), for the real DFT pz(j) = 16 (i / 2) + (q0 ^
        // 8 (i mod 2) ^ (i ^ i / 8) mod 8).
        const int t = fresh(), x = INV ? t & (N - 1) : (t & (HALF - 1)) + HALF * f;
        const int b = INV ? opaque(LR::byte(r0, x < n ? C::out(KIND, x + o) : 0))
                          : opaque(LC::byte(t & (HALF - 1), q0));
        auto from = [&](const int i) {
            if constexpr (INV) return b + RR * i * PB;
            else return (b ^ (4 * ((8 * (i & 1)) ^ (KIND == kDst ? i >> 1 : (i ^ (i >> 3)) & 7)))) + 64 * (i >> 1);
        };
        auto lane = [&](const int i, const int es) {
            if constexpr (INV) return row_lane(x, es);
            else if (i > 0) return col_lane(x, es);
            else return x < n && q0 >= o ? ((q0 - o) * n + x) * es : (int)pts * es;
        };
        auto so = [&](const int i, const int es) {
            if constexpr (INV) return row_so(f, i, es);
            else return i == 0 ? 0 : (CR * i - o) * n * es;
        };
        constexpr int KB = 16;   // elements in flight
#pragma unroll
        for (int i0 = 0; i0 < II; i0 += KB) {
            Tout old[KB];
            float r[KB];
#pragma unroll
            for (int e = 0; e < KB; ++e) {
                const int i = i0 + e;
                if constexpr (ACC == 1) old[e] = dst.load(lane(i, sizeof(Tout)), so(i, sizeof(Tout)));
                if constexpr (ACC == 2) old[e] = (Tout)bp.load(lane(i, 4), so(i, 4));
            }
#pragma unroll
            for (int e = 0; e < KB; ++e) r[e] = at(from(i0 + e));
#pragma unroll
            for (int e = 0; e < KB; ++e) {
                const int i = i0 + e;
                const Tout val = ACC == 0 ? (Tout)r[e] : (Tout)(old[e] + (Tout)r[e]);
                dst.store(val, lane(i, sizeof(Tout)), so(i, sizeof(Tout)));
            }
        }
        if constexpr (f == 0) __syncthreads();   // every thread has read the half
    });
    if (reset && blockIdx.x == 0 && tid == 0) reset[p] = 0;
}

template <typename Tin, typename Tout, int ACC, int KIND, bool INV>
static hipError_t plane_reg_k(const PlaneArgs& a) {
    auto k = plane_reg_kernel<Tin, Tout, ACC, KIND, INV>;
    const size_t lds = PlaneRegCfg::lds_bytes();
    hipError_t e = allow_lds(k, lds);
    if (e != hipSuccess) return e;
    const BatchPtr<const Tin> in{(const Tin*)a.in, a.in_tab, a.bs_in};
    const BatchPtr<Tout> out{(Tout*)a.out, a.out_tab, a.bs_out};
    hipLaunchKernelGGL(k, dim3(a.nplanes, a.batch), dim3(PlaneRegCfg::NT), lds, a.stream, in, out,
                       (float)(INV ? a.sy : a.sx), (float)(INV ? a.sx : a.sy), (const float*)a.tables, a.done, a.base,
                       a.bs_out, a.reset);
    return hipGetLastError();
}

template <typename Tin, typename Tout>
hipError_t launch_plane_reg(const PlaneArgs& a) {
    if (a.stream_planes || (a.base && !a.accum)) return hipErrorInvalidValue;
    if (a.kind == kDst) {
        if constexpr (std::is_same_v<Tin, float>) {
            if (a.inverse) {
                if constexpr (std::is_same_v<Tout, double>) {
                    if (a.base) return plane_reg_k<Tin, Tout, 2, kDst, true>(a);
                    if (a.accum) return plane_reg_k<Tin, Tout, 1, kDst, true>(a);
                }
                if (a.base || a.accum) return hipErrorInvalidValue;
                return plane_reg_k<Tin, Tout, 0, kDst, true>(a);
            }
        }
        if constexpr (std::is_same_v<Tout, float>) {
            if (a.inverse || a.base || a.accum) return hipErrorInvalidValue;
            return plane_reg_k<Tin, Tout, 0, kDst, false>(a);
        }
        return hipErrorInvalidValue;
    }
    if constexpr (std::is_same_v<Tin, float> && std::is_same_v<Tout, float>) {
        if (a.base || a.accum) return hipErrorInvalidValue;
        if (a.kind == kRdftFwd) return plane_reg_k<Tin, Tout, 0, kRdftFwd, false>(a);
        if (a.kind == kRdftInv) return plane_reg_k<Tin, Tout, 0, kRdftInv, true>(a);
    }
    return hipErrorInvalidValue;
}

template hipError_t launch_plane_reg<float, float>(const PlaneArgs&);
template hipError_t launch_plane_reg<double, float>(const PlaneArgs&);
template hipError_t launch_plane_reg<float, double>(const PlaneArgs&);

}  // namespace fdmgpu
