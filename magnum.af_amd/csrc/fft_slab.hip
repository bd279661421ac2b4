// The y and z stages of the zero-padded demag convolution of films of a few layers in one pass: a
// work-group takes one column kx of all layers and components from the x half spectrum through the
// forward y and z transforms, the tensor product and both inverses, in place.
//
// The separate passes are bound by memory, and most of what they move is the spectrum padded along
// y, written and read twice: at 1024 x 1024 x 4 FP32 y forward 302, z and product 529 and y inverse
// 302 MB, where the column pass reads and writes 100 MB each and the tensor once.
//
// ky of a column of N = ny rows (padded to 2 N) is split into S classes ky = S k + r, k < Q = 2 N / S:
//   X[S k + r] = FFT_Q(a_r)[k],  a_r[n] = w_2N^(r n) sum_p w_S^(r p) x[n + Q p],  p < S / 2,
//   y[n + Q p] = sum_r w_S^(-r p) w_2N^(-r n) IFFT_Q(H_r)[n],
// so that one class of all 3 nz lines is in LDS at a time.  Eight values per lane: Q / 8 lanes own a
// line, which never leaves its wave within a class's transform, so its stages are separated by the
// order of the wave's own LDS accesses; the group meets only around the tensor product.  Inputs and
// outputs of a class sit at n = j + (Q / 8) q of lane j, the same for every class: the column stays in
// registers (KEEP) or is read again per class from the caches, and the output sums stay in registers.
//
// FP32: the tensor rows of a pair of mirror classes, r and S - r, are the same; each class loads them while it
// is transformed (the second from the caches) and stages them in LDS, so that no k-point waits for them.  FP64 (the complex
// tensor, 1.6 GB at 1024 x 1024 x 4) and 8 layers: the z transform of a k-point runs on two neighbouring
// lanes, one for the even and one for the odd kz, which halves the registers it needs; their inverses are
// added across the pair.
//
// At 1024 x 1024 x 4 FP32 the pass takes 183 us (the three it replaces 219) and moves 357 MB, 71 us at
// the copy rate; vector instructions take 80 us and LDS 70 us, and one group of 12 waves per CU overlaps
// them little.  80 registers and two groups per CU (the column read again per class) spill and take twice
// as long.  FP64: 699 us against 850, bound by the tensor's bytes (320 us) and the latency of its loads.
#include <hip/hip_runtime.h>

#include "fft_kernels.hpp"
#include "fft_mixed.hpp"
#include "mafx_internal.hpp"

namespace mafx {

namespace {

constexpr int kSlabShared = 2; // columns of a last round that several groups share, at most
constexpr int kSlabPad = 16; // tensor entries between classes 0 (k <= Q / 2) and S / 2

template <class C, int NZ, int LOGN, int LOGS> struct SlabShape {
    static constexpr bool F64 = sizeof(C) == sizeof(double2);
    static constexpr int N = 1 << LOGN, S = 1 << LOGS, LOGQ = LOGN + 1 - LOGS, Q = 1 << LOGQ;
    static constexpr int LPL = Q / 8, LPW = 64 / LPL;               // lanes per line, lines per wave
    static constexpr int NL = 3 * NZ, WAVES = (NL + LPW - 1) / LPW; // lines, waves
    static constexpr int BS = 64 * WAVES, REG = Q + Q / 8, P = S / 2, R3 = Q / 64;
    static constexpr int DATA = WAVES * LPW * REG, TW = 2 * N + 64 + (R3 > 1 ? 64 * R3 : 0); // complex values
    static constexpr int ROW = Q + kSlabPad, TENS = F64 ? 0 : 6 * (NZ + 1) * ROW;            // staged tensor, reals
    static constexpr int TV = (TENS / 4 + BS - 1) / BS;                                      // its float4 per lane
    static constexpr size_t LDS = (static_cast<size_t>(DATA) + TW) * sizeof(C) + TENS * sizeof(float);
    static_assert(LOGQ >= 6 && LOGQ <= 9 && BS <= 1024, "a line is at most one wave");
};

using f32x4 = __attribute__((ext_vector_type(4))) float;

// LDS accesses of one wave execute in order; this keeps the compiler from moving them across
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// keeps the scheduler from starting the next piece's reads early, for which no registers are free
__device__ __forceinline__ void hold_order() { __builtin_amdgcn_sched_barrier(0); }

// the other lane of the pair (lane ^ 1)
__device__ __forceinline__ int pair_int(int v) { return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true); }
__device__ __forceinline__ float pair_get(float v) { return __int_as_float(pair_int(__float_as_int(v))); }
__device__ __forceinline__ double pair_get(double v) {
    return __hiloint2double(pair_int(__double2hiint(v)), pair_int(__double2loint(v)));
}

// exp(-2 pi i k / (2 NZ))
template <class C, int NZ> __device__ __forceinline__ C zroot(int k) {
    using T = typename real_of<C>::type;
    constexpr int R = NZ == 3 ? 6 : NZ == 5 ? 10 : 16, step = R / (2 * NZ);
    return C{static_cast<T>(Root<R>::c[k * step]), static_cast<T>(-Root<R>::s[k * step])};
}

// FFT_Q of a line: v holds positions j + LPL q on entry and on return; lb is the line's LDS region,
// position i at i + i / 8, which spreads the writes at strides 8 and 64 over the banks and keeps every
// access one address and constant offsets.  t2[8 q + k] = w_64^(q k), t3[64 r + b] = w_Q^(r b).
template <class C, class SH, bool INV>
__device__ __forceinline__ void slab_fft(C (&v)[8], C* lb, const C* t2, const C* t3, int j) {
    constexpr int LPL = SH::LPL, R3 = SH::R3, RS = LPL + LPL / 8;
    const int k = j & 7;
    C *rd = lb + j + (j >> 3), *w1 = lb + 9 * j, *w2 = lb + 9 * (j - k) + k;
    dft<C, 8>(v, INV, t2, 8);
    wave_order();
#pragma unroll
    for (int q = 0; q < 8; ++q) w1[q] = v[q];
    wave_order();
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = rd[RS * q];
#pragma unroll
    for (int q = 1; q < 8; ++q) v[q] = cmul(v[q], conj_if(t2[8 * q + k], INV));
    dft<C, 8>(v, INV, t2, 8);
    if constexpr (R3 > 1) {
        wave_order();
#pragma unroll
        for (int q = 0; q < 8; ++q) w2[9 * q] = v[q];
        wave_order();
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = rd[RS * q];
        constexpr int G = 8 / R3; // butterflies per lane
#pragma unroll
        for (int i = 0; i < G; ++i) {
            C u[R3];
#pragma unroll
            for (int r = 0; r < R3; ++r) u[r] = r == 0 ? v[i] : cmul(v[i + r * G], conj_if(t3[64 * r + j + LPL * i], INV));
            dft<C, R3>(u, INV, t2, R3);
#pragma unroll
            for (int r = 0; r < R3; ++r) v[i + r * G] = u[r];
        }
    }
}

// Tensor rows: FP64 [kx][r][6][2 NZ][Q], complex; FP32 [kx][r <= S / 2 - 1][6][NZ + 1][Q + kSlabPad], real,
// one block for each pair of mirror classes: r and S - r, or 0 (k <= Q / 2) and S / 2 (k < Q / 2).
template <class SH> __device__ __forceinline__ void slab_row(int r, int k, int& at, float& sy) {
    constexpr int Q = SH::Q, S = SH::S;
    if (r == 0) {
        sy = k <= Q / 2 ? 1.0f : -1.0f;
        at = k <= Q / 2 ? k : Q - k;
    } else if (2 * r == S) {
        sy = k < Q / 2 ? 1.0f : -1.0f;
        at = Q / 2 + kSlabPad + (k < Q / 2 ? k : Q - 1 - k);
    } else {
        sy = 2 * r > S ? -1.0f : 1.0f;
        at = 2 * r > S ? Q - 1 - k : k;
    }
}
template <int NZ, int ROW>
__device__ __forceinline__ void sym_product(float2& X0, float2& X1, float2& X2, const float* t, int kz, float sy) {
    constexpr int NH = NZ + 1;
    const float sz = kz <= NZ ? 1.0f : -1.0f;
    const float* tz = t + (kz <= NZ ? kz : 2 * NZ - kz) * ROW;
    const float xx = tz[0], xy = sy * tz[NH * ROW], xz = sz * tz[2 * NH * ROW], yy = tz[3 * NH * ROW],
                yz = sy * sz * tz[4 * NH * ROW], zz = tz[5 * NH * ROW];
    const float2 a = X0, b = X1, d = X2;
    X0 = float2{xx * a.x + xy * b.x + xz * d.x, xx * a.y + xy * b.y + xz * d.y};
    X1 = float2{xy * a.x + yy * b.x + yz * d.x, xy * a.y + yy * b.y + yz * d.y};
    X2 = float2{xz * a.x + yz * b.x + zz * d.x, xz * a.y + yz * b.y + zz * d.y};
}

template <class C, int NZ, int LOGN, int LOGS, bool KEEP>
__global__ void __launch_bounds__((SlabShape<C, NZ, LOGN, LOGS>::BS))
    k_slab(C* __restrict__ spec, int64_t plane, const void* __restrict__ tens, const C* __restrict__ twL, int hx, int nsplit,
           C* part, int* count) {
    using SH = SlabShape<C, NZ, LOGN, LOGS>;
    using T = typename real_of<C>::type;
    constexpr int Q = SH::Q, S = SH::S, P = SH::P, LPL = SH::LPL, NL = SH::NL, REG = SH::REG, N2 = 2 * SH::N, R3 = SH::R3;
    constexpr bool F64 = SH::F64, PAIR = F64 || NZ > 4;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    C *buf = reinterpret_cast<C*>(smem_raw), *tw = buf + SH::DATA, *t2 = tw + N2, *t3 = t2 + 64;
    float* ts = reinterpret_cast<float*>(tw + SH::TW);
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, j0 = lane % LPL;
    const int line = (tid >> 6) * SH::LPW + lane / LPL; // c NZ + z
    // The first nsplit S groups take one class each of the last nsplit columns (slab_rows), the others a
    // column each.
    const int bid = static_cast<int>(blockIdx.x), nfirst = nsplit * S;
    const bool shared = bid < nfirst;
    const int mine = shared ? bid % S : 0;
    const int kx = shared ? hx - nsplit + bid / S
                       : static_cast<int>(xcd_swizzle(static_cast<uint32_t>(bid - nfirst), gridDim.x - static_cast<uint32_t>(nfirst)));
    const int s_end = shared ? mine + 1 : S;
    for (int t = tid; t < N2; t += SH::BS) tw[t] = twL[t];
    for (int t = tid; t < 64; t += SH::BS) t2[t] = twL[(t >> 3) * (t & 7) * (N2 / 64)];
    if constexpr (R3 > 1)
        for (int t = tid; t < 64 * R3; t += SH::BS) t3[t] = twL[S * (t >> 6) * (t & 63)];
    // the lane's part of its line, formed anew where it is used: its addresses are not held meanwhile
    const auto column = [&] {
        const int l = opaque_int(line < NL ? line : NL - 1);
        return spec + l * plane + tcol(kx, static_cast<int64_t>(kTile) * N2) + kTile * j0;
    };
    C* lb = buf + line * REG;
    C x[P][8], acc[P][8];
    const auto load = [&] {
        const C* col = column();
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int q = 0; q < 8; ++q) x[p][q] = col[kTile * (LPL * q + Q * p)];
    };
    if constexpr (KEEP) load();
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < 8; ++q) acc[p][q] = C{0, 0};
    __syncthreads(); // the twiddles
    // mirror classes r and S - r, whose tensor rows are the same, one after the other
#pragma unroll 1
    for (int s = mine; s < s_end; ++s) {
        const int r = s < 2 ? s * (S / 2) : (s & 1) ? S - s / 2 : s / 2;
        const int j = opaque_int(j0); // the stages' addresses are formed per class, not held across it
        f32x4 tv[F64 ? 1 : SH::TV];
        if constexpr (!F64) {
            // the pair's tensor rows, on their way while the class is transformed
            const f32x4* src = reinterpret_cast<const f32x4*>(
                static_cast<const float*>(tens) + (static_cast<int64_t>(kx) * P + s / 2) * SH::TENS);
#pragma unroll
            for (int i = 0; i < SH::TV; ++i) {
                const int e = tid + i * SH::BS;
                tv[i] = src[e < SH::TENS / 4 ? e : 0];
            }
        }
        C ws[P]; // w_S^(r p)
#pragma unroll
        for (int p = 0; p < P; ++p) ws[p] = tw[(r * p * Q) & (N2 - 1)];
        C v[8];
        if constexpr (!KEEP) load();
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            v[q] = x[0][q];
#pragma unroll
            for (int p = 1; p < P; ++p) v[q] = cadd(v[q], cmul(x[p][q], ws[p]));
            if (r > 0) v[q] = cmul(v[q], tw[r * (j + LPL * q)]);
            if (q & 1) hold_order();
        }
        slab_fft<C, SH, false>(v, lb, t2, t3, j);
        wave_order();
        C* const rd = lb + j + (j >> 3);
#pragma unroll
        for (int q = 0; q < 8; ++q) rd[(LPL + LPL / 8) * q] = v[q];
        if constexpr (!F64) {
#pragma unroll
            for (int i = 0; i < SH::TV; ++i) {
                const int e = tid + i * SH::BS;
                if (e < SH::TENS / 4) reinterpret_cast<f32x4*>(ts)[e] = tv[i];
            }
        }
        __syncthreads();
        if constexpr (!PAIR) {
            for (int k = opaque_int(tid); k < Q; k += SH::BS) {
                C* const b = buf + k + (k >> 3);
                int at;
                float sy;
                slab_row<SH>(r, k, at, sy);
                C ev[3][NZ], od[3][NZ];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
#pragma unroll
                    for (int z = 0; z < NZ; ++z) {
                        ev[c][z] = b[(c * NZ + z) * REG];
                        od[c][z] = z > 0 ? cmul(ev[c][z], zroot<C, NZ>(z)) : ev[c][z];
                    }
                    mdft<C, NZ, false>(ev[c]);
                    mdft<C, NZ, false>(od[c]);
                    hold_order();
                }
#pragma unroll
                for (int z = 0; z < NZ; ++z) {
                    sym_product<NZ, SH::ROW>(ev[0][z], ev[1][z], ev[2][z], ts + at, 2 * z, sy);
                    sym_product<NZ, SH::ROW>(od[0][z], od[1][z], od[2][z], ts + at, 2 * z + 1, sy);
                    hold_order();
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    mdft<C, NZ, true>(ev[c]);
                    mdft<C, NZ, true>(od[c]);
#pragma unroll
                    for (int z = 0; z < NZ; ++z)
                        b[(c * NZ + z) * REG] = cadd(ev[c][z], z > 0 ? cmul(od[c][z], conj_if(zroot<C, NZ>(z), true)) : od[c][z]);
                    hold_order();
                }
            }
        } else {
            for (int e = opaque_int(tid); e < 2 * Q; e += SH::BS) { // k-point k, kz of one parity
                const int par = e & 1, k = e >> 1;
                C* const b = buf + k + (k >> 3);
                C h[3][NZ];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
#pragma unroll
                    for (int z = 0; z < NZ; ++z) {
                        h[c][z] = b[(c * NZ + z) * REG];
                        const C w = zroot<C, NZ>(z);
                        if (z > 0) h[c][z] = cmul(h[c][z], C{par ? w.x : T(1), par ? w.y : T(0)});
                    }
                    mdft<C, NZ, false>(h[c]);
                    hold_order();
                }
                if constexpr (F64) {
                    const C* t = static_cast<const C*>(tens) + (static_cast<int64_t>(kx) * S + r) * (12 * NZ * Q) + par * Q + k;
#pragma unroll
                    for (int z = 0; z < NZ; ++z) {
                        const C* tz = t + 2 * z * Q;
                        const C xx = tz[0], xy = tz[2 * NZ * Q], xz = tz[4 * NZ * Q], yy = tz[6 * NZ * Q],
                                yz = tz[8 * NZ * Q], zz = tz[10 * NZ * Q];
                        const C a = h[0][z], b1 = h[1][z], d = h[2][z];
                        h[0][z] = cadd(cadd(cmul(xx, a), cmul(xy, b1)), cmul(xz, d));
                        h[1][z] = cadd(cadd(cmul(xy, a), cmul(yy, b1)), cmul(yz, d));
                        h[2][z] = cadd(cadd(cmul(xz, a), cmul(yz, b1)), cmul(zz, d));
                        if (z & 1) hold_order();
                    }
                } else {
                    int at;
                    float sy;
                    slab_row<SH>(r, k, at, sy);
#pragma unroll
                    for (int z = 0; z < NZ; ++z) {
                        sym_product<NZ, SH::ROW>(h[0][z], h[1][z], h[2][z], ts + at, 2 * z + par, sy);
                        hold_order();
                    }
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    mdft<C, NZ, true>(h[c]);
#pragma unroll
                    for (int z = 0; z < NZ; ++z) {
                        const C w = zroot<C, NZ>(z);
                        if (z > 0) h[c][z] = cmul(h[c][z], C{par ? w.x : T(1), par ? -w.y : T(0)});
                        h[c][z] = C{h[c][z].x + pair_get(h[c][z].x), h[c][z].y + pair_get(h[c][z].y)};
                    }
                    hold_order();
                }
                // the pair's lanes, which have read position k, store every other line of it
#pragma unroll
                for (int i = 0; i < NL; i += 2) {
                    const C v0 = h[i / NZ][i % NZ], v1 = i + 1 < NL ? h[(i + 1) / NZ % 3][(i + 1) % NZ] : v0;
                    if (i + 1 < NL || par == 0) b[(i + par) * REG] = C{par ? v1.x : v0.x, par ? v1.y : v0.y};
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = rd[(LPL + LPL / 8) * q];
        slab_fft<C, SH, true>(v, lb, t2, t3, j);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            if (r > 0) v[q] = cmul(v[q], conj_if(tw[r * (j + LPL * q)], true));
            acc[0][q] = cadd(acc[0][q], v[q]);
#pragma unroll
            for (int p = 1; p < P; ++p) acc[p][q] = cadd(acc[p][q], cmul(v[q], conj_if(ws[p], true)));
            if (q & 1) hold_order();
        }
    }
    if (shared) {
        // the group that finishes a column last adds the groups' sums in their order
        int* last = reinterpret_cast<int*>(tw); // the twiddles are done with
        constexpr int PER = P * 8 * SH::BS;     // values of one group
        const int at = kx - (hx - nsplit);
        C* sums = part + static_cast<int64_t>(at) * S * PER + tid;
#pragma unroll
        for (int i = 0; i < P * 8; ++i) sums[mine * PER + i * SH::BS] = acc[i / 8][i % 8];
        __threadfence();
        __syncthreads();
        if (tid == 0) {
            *last = atomicAdd(count + at, 1) == S - 1;
            if (*last) count[at] = 0; // for the next launch
        }
        __syncthreads();
        if (!*last) return;
        __threadfence();
#pragma unroll
        for (int i = 0; i < P * 8; ++i) {
            C v = sums[i * SH::BS];
#pragma unroll
            for (int g = 1; g < S; ++g) v = cadd(v, sums[g * PER + i * SH::BS]);
            acc[i / 8][i % 8] = v;
        }
    }
    if (line < NL) {
        C* col = column();
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int q = 0; q < 8; ++q) col[kTile * (LPL * q + Q * p)] = acc[p][q];
    }
}

// ---- tensor rows -------------------------------------------------------------------------------
__global__ void k_slab_rows_f64(const double2* __restrict__ T, double2* __restrict__ out, int64_t total, int planes, int S,
                                int Q, int64_t plane) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= total) return;
    const int k = static_cast<int>(e % Q);
    const int64_t a = e / Q, b = a / planes, kx = b / S;
    const int p = static_cast<int>(a - b * planes), r = static_cast<int>(b - kx * S);
    out[e] = T[p * plane + tcol(kx, static_cast<int64_t>(kTile) * S * Q) + static_cast<int64_t>(kTile) * (S * k + r)];
}
__global__ void k_slab_rows_f32(const float* __restrict__ T, float* __restrict__ out, int64_t total, int planes, int S,
                                int Q, int64_t plane) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= total) return;
    const int N = S * Q / 2, row = Q + kSlabPad, i = static_cast<int>(e % row);
    const int64_t a = e / row, b = a / planes, kx = b / (S / 2);
    const int p = static_cast<int>(a - b * planes), r = static_cast<int>(b - kx * (S / 2));
    int ky;
    if (r > 0)
        ky = i < Q ? S * i + r : -1;
    else if (i < Q / 2 + kSlabPad)
        ky = i <= Q / 2 ? S * i : -1;
    else
        ky = S * (i - Q / 2 - kSlabPad) + S / 2;
    // the stored quarter holds ky <= N; xy and yz are odd in ky
    const int c = 6 * p / planes;
    const float sign = ky > N && (c == 1 || c == 4) ? -1.0f : 1.0f;
    if (ky > N) ky = 2 * N - ky;
    out[e] = ky < 0 ? 0.0f : sign * T[p * plane + tcol(kx, static_cast<int64_t>(kTile) * (N + 1)) + static_cast<int64_t>(kTile) * ky];
}

template <class C> using SlabFn = void (*)(C*, int64_t, const void*, const C*, int, int, C*, int*);
template <class C> struct SlabPlan {
    SlabFn<C> fn{nullptr};
    int S{0}, Q{0}, block{0};
    size_t lds{0};
};
template <class C, int NZ, int LOGN> SlabPlan<C> slab_plan_of() {
    // the fewest classes whose lines are one wave and whose group has at most 12 waves; FP64 columns are
    // read again per class (the sums alone take 64 registers)
    constexpr int LOGS = LOGN == 10 || (LOGN == 9 && NZ > 4) ? 2 : 1;
    constexpr bool KEEP = sizeof(C) == sizeof(float2);
    using SH = SlabShape<C, NZ, LOGN, LOGS>;
    return {k_slab<C, NZ, LOGN, LOGS, KEEP>, SH::S, SH::Q, SH::BS, SH::LDS};
}
// Films of 2, 3, 4 or 8 layers of a power of two of rows, 64 to 1024; 5, 6 and 7 layers have no kernel here
// and were not measured.  A group has a CU to itself where its LDS or registers fill one (`heavy`), so the
// pass takes as long as its rounds of columns, while the separate passes follow the bytes.  It is left out
// where they were faster, demag field evaluations in us, separate passes against column pass on 256 CUs:
// - no kernel: the sums do not fit the registers.  FP32 1024 x 1024 x 8 742, 915; FP64 512 x 512 x 8 500, 632;
// - long columns that leave CUs idle.  FP32 100 x 512 x 8 71, 77; FP64 100 x 1024 x 4 132, 159, 64 x 512 x 3
//   50, 51;
// - heavy columns whose last round is nearly empty.  FP32 260 x 1024 x 2 76, 90; FP64 260 x 256 x 3 73, 83;
// - the two shapes that gain least: FP32 1024 x 2 layers unless nine tenths of the rounds are filled
//   (600 columns 139, 148; 800 179, 195; 1000 is 2 % faster), and FP64 256 x 3 layers from 3 to 8 rounds
//   (800 200, 212; 1024 190, 194; 500 is 20 %, 2048 4 % faster).
// Elsewhere, over 64 to 2048 columns, it is 2 % slower to 83 % faster: FP32 512 x 64 x 4 44, 26; 1024 x 256 x 2
// 67, 49; 512 x 512 x 4 100, 90; 1024 x 1024 x 4 353, 302; FP64 512 x 128 x 2 55, 36; 512 x 512 x 4 249, 218;
// 1024 x 1024 x 4 1050, 883.
template <class C> SlabPlan<C> slab_plan(int nx, int ny, int nz, int cus) {
    constexpr bool F64 = sizeof(C) == sizeof(double2);
    const int hx = nx + 1, rounds = (hx + cus - 1) / cus;
    const bool heavy = ny == 1024 || (ny == 512 && nz == 8) || (F64 && ny == 256 && nz > 2);
    if (nx < cus && (ny == 1024 ? F64 || nz == 4 || 3 * nx < cus : ny == 512 && (nz == 8 || (F64 && nz > 2 && 3 * nx < cus))))
        return {};
    // a last round of up to kSlabShared columns is spread over the other rounds (slab_rows)
    const bool partly = rounds > 1 && hx % cus > kSlabShared;
    if (heavy && partly && 4 * hx < 3 * rounds * cus) return {};
    if (!F64 && ny == 1024 && nz == 2 && partly && 10 * hx < 9 * rounds * cus) return {};
    if (F64 && ny == 256 && nz == 3 && hx > 3 * cus && hx < 8 * cus) return {};
    switch (100 * ny + nz) {
#define MAFX_SLAB(NZ, LOGN) \
    case 100 * (1 << LOGN) + NZ: return slab_plan_of<C, NZ, LOGN>();
#define MAFX_SLAB_ROWS(LOGN) MAFX_SLAB(2, LOGN) MAFX_SLAB(3, LOGN) MAFX_SLAB(4, LOGN)
        MAFX_SLAB_ROWS(6)
        MAFX_SLAB_ROWS(7)
        MAFX_SLAB_ROWS(8)
        MAFX_SLAB_ROWS(9)
        MAFX_SLAB_ROWS(10)
        MAFX_SLAB(8, 6)
        MAFX_SLAB(8, 7)
#undef MAFX_SLAB_ROWS
#undef MAFX_SLAB
    default: break;
    }
    if constexpr (!F64) {
        if (nz == 8 && ny == 256) return slab_plan_of<C, 8, 8>();
        if (nz == 8 && ny == 512) return slab_plan_of<C, 8, 9>();
    }
    return {};
}

template <class C> SlabPlan<C> plan_of(const mafx_ctx* ctx) {
    const mafx_mesh& g = ctx->mesh;
    if (g.nx > (1 << 24) || g.ny > 1024 || g.nz > 8) return {};
    return slab_plan<C>(static_cast<int>(g.nx), static_cast<int>(g.ny), static_cast<int>(g.nz), ctx->num_cus);
}

template <class C> void slab_run(mafx_ctx* ctx, C* spec, const void* t) {
    const SlabPlan<C> p = plan_of<C>(ctx);
    const int64_t plane = ctx->n1 * ctx->hxs;
    ProfScope ps(ctx, sizeof(C) == sizeof(float2) ? "slab_f32" : "slab_f64",
                 6.0 * static_cast<double>(ctx->mesh.nz * ctx->mesh.ny * ctx->hx) * sizeof(C) + static_cast<double>(ctx->tensor.bytes));
    const int hx = static_cast<int>(ctx->hx), ns = ctx->slab_split;
    hipLaunchKernelGGL(p.fn, dim3(static_cast<unsigned>(hx + ns * (p.S - 1))), dim3(p.block), p.lds, ctx->stream, spec, plane,
                       t, tw_of<C>(ctx->py), hx, ns, ctx->slab_part.as<C>(), ctx->slab_count.as<int>());
    MAFX_HIP(hipGetLastError());
}

template <class C> void slab_rows(mafx_ctx* ctx) {
    const SlabPlan<C> p = plan_of<C>(ctx);
    if (!p.fn) return;
    MAFX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(p.fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(p.lds)));
    constexpr bool F64 = sizeof(C) == sizeof(double2);
    const int planes = static_cast<int>(F64 ? 6 * ctx->n2 : 6 * ctx->n2h);
    const int64_t total = F64 ? ctx->hx * p.S * planes * p.Q : ctx->hx * (p.S / 2) * planes * (p.Q + kSlabPad);
    DevBuf rows;
    rows.alloc(total * (F64 ? sizeof(double2) : sizeof(float)));
    const dim3 g(grid_for(total, 256)), b(256);
    if constexpr (F64)
        hipLaunchKernelGGL(k_slab_rows_f64, g, b, 0, ctx->stream, ctx->tensor.as<double2>(), rows.as<double2>(), total, planes,
                           p.S, p.Q, ctx->n1 * ctx->hxs);
    else
        hipLaunchKernelGGL(k_slab_rows_f32, g, b, 0, ctx->stream, ctx->tensor.as<float>(), rows.as<float>(), total, planes,
                           p.S, p.Q, ctx->n1h * ctx->hxs);
    MAFX_HIP(hipGetLastError());
    // A group has a CU to itself, and with nx = 2^n the columns are one more than whole rounds of the
    // chip: the one or two columns of a last round are started first, their classes spread over S groups.
    // (1024 x 1024 x 4: 308 -> 302 us in FP32, 937 -> 874 in FP64.  Each sharing group writes its L2 back:
    // with all 101 columns of 100 x 512 x 4 shared the field takes 139 us instead of 44.)
    const int tail = static_cast<int>(ctx->hx % ctx->num_cus);
    ctx->slab_split = ctx->hx > ctx->num_cus && tail <= kSlabShared ? tail : 0;
    if (ctx->slab_split > 0) {
        ctx->slab_part.alloc(sizeof(C) * ctx->slab_split * p.S * (p.S / 2 * 8) * p.block);
        ctx->slab_count.alloc(sizeof(int) * ctx->slab_split);
        MAFX_HIP(hipMemsetAsync(ctx->slab_count.p, 0, ctx->slab_count.bytes, ctx->stream));
    }
    // rows and counters are complete for any stream that the context is given later
    MAFX_HIP(hipStreamSynchronize(ctx->stream));
    ctx->tensor = std::move(rows);
    ctx->slab = true;
}

} // namespace

void slab_prepare(mafx_ctx* ctx) {
    if (ctx->atom_dipole || demag_full_c32(ctx->precision, ctx->demag_flags) || ctx->nzs != ctx->mesh.nz) return;
    if (demag_f64(ctx->precision))
        slab_rows<double2>(ctx);
    else
        slab_rows<float2>(ctx);
}
void slab_column(mafx_ctx* ctx, double2* spec) { slab_run<double2>(ctx, spec, ctx->tensor.p); }
void slab_column(mafx_ctx* ctx, float2* spec) { slab_run<float2>(ctx, spec, ctx->tensor.p); }

} // namespace mafx
