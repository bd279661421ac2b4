// Mixed-radix LDS FFT for lines of any length whose prime factors are at most 13.
//
// Lines lie in LDS as [pos][line], in two buffers: a stage reads one and writes the other (the
// autosort order of fft_device.hpp), so it needs one barrier, a lane runs any number of butterflies
// one after the other with only one butterfly's values in registers, and the register budget does
// not grow with the tile.  That lets the tile follow the problem: small tiles fill the chip on small
// meshes, where the in-place kernels (whose lanes hold all their butterflies across a barrier) ran
// a handful of large groups.  Radices up to 16 keep the number of stages at two or three; they are
// products of register DFTs whose constants are compile-time values.
#pragma once
#include "fft_device.hpp"

namespace mafx {

constexpr int kMixStages = 6;

// Stage schedule of one length: radices in order, Ns (product of the radices before a stage) as a
// divisor, and the twiddle step L / (Ns R).  nstages == 0: the length has no schedule here.
struct MixDesc {
    int L, nstages;
    int radix[kMixStages], twstep[kMixStages];
    FastDiv ns[kMixStages];
};

template <int R> struct Root;
template <> struct Root<3> { // cos, sin of 2 pi k / 3
        static constexpr double c[3] = {1.0, -0.5, -0.5};
        static constexpr double s[3] = {0.0, 0.8660254037844386, -0.8660254037844386};
};
template <> struct Root<5> { // cos, sin of 2 pi k / 5
        static constexpr double c[5] = {1.0, 0.30901699437494745, -0.8090169943749475, -0.8090169943749475,
        0.30901699437494745};
        static constexpr double s[5] = {0.0, 0.9510565162951535, 0.5877852522924731, -0.5877852522924731,
        -0.9510565162951535};
};
template <> struct Root<6> { // cos, sin of 2 pi k / 6
        static constexpr double c[6] = {1.0, 0.5, -0.5, -1.0, -0.5, 0.5};
        static constexpr double s[6] = {0.0, 0.8660254037844386, 0.8660254037844386, 0.0, -0.8660254037844386,
        -0.8660254037844386};
};
template <> struct Root<7> { // cos, sin of 2 pi k / 7
        static constexpr double c[7] = {1.0, 0.6234898018587335, -0.2225209339563144, -0.9009688679024191,
        -0.9009688679024191, -0.2225209339563144, 0.6234898018587335};
        static constexpr double s[7] = {0.0, 0.7818314824680298, 0.9749279121818236, 0.4338837391175581,
        -0.4338837391175581, -0.9749279121818236, -0.7818314824680298};
};
template <> struct Root<9> { // cos, sin of 2 pi k / 9
        static constexpr double c[9] = {1.0, 0.766044443118978, 0.17364817766693036, -0.5, -0.9396926207859084,
        -0.9396926207859084, -0.5, 0.17364817766693036, 0.766044443118978};
        static constexpr double s[9] = {0.0, 0.6427876096865394, 0.984807753012208, 0.8660254037844386,
        0.3420201433256687, -0.3420201433256687, -0.8660254037844386, -0.984807753012208, -0.6427876096865394};
};
template <> struct Root<10> { // cos, sin of 2 pi k / 10
        static constexpr double c[10] = {1.0, 0.8090169943749475, 0.30901699437494745, -0.30901699437494745,
        -0.8090169943749475, -1.0, -0.8090169943749475, -0.30901699437494745, 0.30901699437494745,
        0.8090169943749475};
        static constexpr double s[10] = {0.0, 0.5877852522924731, 0.9510565162951535, 0.9510565162951535,
        0.5877852522924731, 0.0, -0.5877852522924731, -0.9510565162951535, -0.9510565162951535, -0.5877852522924731};
};
template <> struct Root<11> { // cos, sin of 2 pi k / 11
        static constexpr double c[11] = {1.0, 0.8412535328311812, 0.41541501300188644, -0.14231483827328514,
        -0.6548607339452851, -0.9594929736144974, -0.9594929736144974, -0.6548607339452851, -0.14231483827328514,
        0.41541501300188644, 0.8412535328311812};
        static constexpr double s[11] = {0.0, 0.5406408174555976, 0.9096319953545183, 0.9898214418809327,
        0.7557495743542583, 0.28173255684142967, -0.28173255684142967, -0.7557495743542583, -0.9898214418809327,
        -0.9096319953545183, -0.5406408174555976};
};
template <> struct Root<12> { // cos, sin of 2 pi k / 12
        static constexpr double c[12] = {1.0, 0.8660254037844386, 0.5, 0.0, -0.5, -0.8660254037844386, -1.0,
        -0.8660254037844386, -0.5, 0.0, 0.5, 0.8660254037844386};
        static constexpr double s[12] = {0.0, 0.5, 0.8660254037844386, 1.0, 0.8660254037844386, 0.5, 0.0, -0.5,
        -0.8660254037844386, -1.0, -0.8660254037844386, -0.5};
};
template <> struct Root<13> { // cos, sin of 2 pi k / 13
        static constexpr double c[13] = {1.0, 0.8854560256532099, 0.5680647467311558, 0.12053668025532305,
        -0.3546048870425356, -0.7485107481711011, -0.970941817426052, -0.970941817426052, -0.7485107481711011,
        -0.3546048870425356, 0.12053668025532305, 0.5680647467311558, 0.8854560256532099};
        static constexpr double s[13] = {0.0, 0.46472317204376856, 0.8229838658936564, 0.992708874098054,
        0.9350162426854148, 0.6631226582407952, 0.23931566428755777, -0.23931566428755777, -0.6631226582407952,
        -0.9350162426854148, -0.992708874098054, -0.8229838658936564, -0.46472317204376856};
};
template <> struct Root<15> { // cos, sin of 2 pi k / 15
        static constexpr double c[15] = {1.0, 0.9135454576426009, 0.6691306063588582, 0.30901699437494745,
        -0.10452846326765347, -0.5, -0.8090169943749475, -0.9781476007338057, -0.9781476007338057,
        -0.8090169943749475, -0.5, -0.10452846326765347, 0.30901699437494745, 0.6691306063588582, 0.9135454576426009};
        static constexpr double s[15] = {0.0, 0.4067366430758002, 0.7431448254773942, 0.9510565162951535,
        0.9945218953682733, 0.8660254037844386, 0.5877852522924731, 0.20791169081775934, -0.20791169081775934,
        -0.5877852522924731, -0.8660254037844386, -0.9945218953682733, -0.9510565162951535, -0.7431448254773942,
        -0.4067366430758002};
};
template <> struct Root<16> { // cos, sin of 2 pi k / 16
        static constexpr double c[16] = {1.0, 0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0.0,
        -0.3826834323650898, -0.7071067811865476, -0.9238795325112867, -1.0, -0.9238795325112867, -0.7071067811865476,
        -0.3826834323650898, 0.0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867};
        static constexpr double s[16] = {0.0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867, 1.0,
        0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0.0, -0.3826834323650898, -0.7071067811865476,
        -0.9238795325112867, -1.0, -0.9238795325112867, -0.7071067811865476, -0.3826834323650898};
};

template <class C> __device__ __forceinline__ C rot(C a, double c, double s, bool inv) { // a exp(-+ i t), c + i s = exp(i t)
    using T = typename real_of<C>::type;
    return cmul(a, C{static_cast<T>(c), static_cast<T>(inv ? s : -s)});
}

// R-point DFT in registers, forward (exp(-2 pi i / R)) or inverse.
template <class C, int R, bool INV> __device__ __forceinline__ void mdft(C (&v)[R]);

// R = A B: length-A transforms over n1 of v[B n1 + n2], twiddles w_R^(n2 k1), length-B transforms
// over n2; output k1 + A k2.
template <class C, int A, int B, bool INV> __device__ __forceinline__ void mdft2(C (&v)[A * B]) {
    constexpr int R = A * B;
    C y[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) y[n2][n1] = v[B * n1 + n2];
        mdft<C, A, INV>(y[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        C x[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2)
            x[n2] = n2 * k1 == 0 ? y[n2][k1] : rot(y[n2][k1], Root<R>::c[n2 * k1], Root<R>::s[n2 * k1], INV);
        mdft<C, B, INV>(x);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = x[k2];
    }
}

template <class C, int R, bool INV> __device__ __forceinline__ void mdft(C (&v)[R]) {
    using T = typename real_of<C>::type;
    if constexpr (R == 2 || R == 4 || R == 8) {
        dft<C, R>(v, INV, static_cast<const C*>(nullptr), R);
    } else if constexpr (R == 3 || R == 5 || R == 7 || R == 11 || R == 13) {
        // pairs j, R - j: sums meet the cosines, differences the sines
        constexpr int H = R / 2;
        C a[H], b[H], out[R];
        out[0] = v[0];
#pragma unroll
        for (int j = 0; j < H; ++j) {
            a[j] = cadd(v[j + 1], v[R - 1 - j]);
            b[j] = csub(v[j + 1], v[R - 1 - j]);
            out[0] = cadd(out[0], a[j]);
        }
#pragma unroll
        for (int q = 1; q <= H; ++q) {
            C t = v[0], u{0, 0};
#pragma unroll
            for (int j = 0; j < H; ++j) {
                const T c = static_cast<T>(Root<R>::c[((j + 1) * q) % R]), s = static_cast<T>(Root<R>::s[((j + 1) * q) % R]);
                t = C{t.x + c * a[j].x, t.y + c * a[j].y};
                u = C{u.x + s * b[j].x, u.y + s * b[j].y};
            }
            const C m = mul_mi(u, INV); // -i u forward, +i u inverse
            out[q] = cadd(t, m);
            out[R - q] = csub(t, m);
        }
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = out[q];
    } else if constexpr (R == 6) {
        mdft2<C, 2, 3, INV>(v);
    } else if constexpr (R == 9) {
        mdft2<C, 3, 3, INV>(v);
    } else if constexpr (R == 10) {
        mdft2<C, 2, 5, INV>(v);
    } else if constexpr (R == 12) {
        mdft2<C, 4, 3, INV>(v);
    } else if constexpr (R == 15) {
        mdft2<C, 3, 5, INV>(v);
    } else {
        static_assert(R == 16, "radices 2..13, 15, 16 without 14");
        mdft2<C, 4, 4, INV>(v);
    }
}

// One stage over `lines` lines: butterfly b = j lines + line reads positions j + r L/R (element
// b + r nb) and writes positions (j / Ns) Ns R + j % Ns + r Ns.
template <class C, int R, bool INV>
__device__ __forceinline__ void mix_stage(const C* src, C* dst, int nb, int lines, const FastDiv& lined,
                                          const FastDiv& Ns, int twstep, const C* __restrict__ tw) {
    const int ns = static_cast<int>(Ns.d), os = ns * lines;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        C v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = src[lds_pad(b + r * nb)];
        const int j = static_cast<int>(fdiv(b, lined)), q = static_cast<int>(fdiv(j, Ns)), step = (j - q * ns) * twstep;
        if (ns > 1) {
#pragma unroll
            for (int r = 1; r < R; ++r) v[r] = cmul(v[r], conj_if(tw[r * step], INV));
        }
        mdft<C, R, INV>(v);
        const int o = b + q * os * (R - 1);
#pragma unroll
        for (int r = 0; r < R; ++r) dst[lds_pad(o + r * os)] = v[r];
    }
}

// All stages of `lines` lines held in a (complete before the call); the result is in the returned
// buffer, a or b, complete for every lane.
template <class C, bool INV>
__device__ C* mix_fft(C* a, C* b, const MixDesc& d, int lines, const FastDiv& lined, const C* __restrict__ tw) {
    for (int s = 0; s < d.nstages; ++s) {
        const int R = d.radix[s], nb = d.L / R * lines, ts = d.twstep[s];
        switch (R) {
#define MAFX_MIX_STAGE(N) \
    case N: mix_stage<C, N, INV>(a, b, nb, lines, lined, d.ns[s], ts, tw); break;
            MAFX_MIX_STAGE(2)
            MAFX_MIX_STAGE(3)
            MAFX_MIX_STAGE(4)
            MAFX_MIX_STAGE(5)
            MAFX_MIX_STAGE(6)
            MAFX_MIX_STAGE(7)
            MAFX_MIX_STAGE(8)
            MAFX_MIX_STAGE(9)
            MAFX_MIX_STAGE(10)
            MAFX_MIX_STAGE(11)
            MAFX_MIX_STAGE(12)
            MAFX_MIX_STAGE(13)
            MAFX_MIX_STAGE(15)
            MAFX_MIX_STAGE(16)
#undef MAFX_MIX_STAGE
        default: break; // unreachable: mix_desc uses these radices only
        }
        __syncthreads();
        C* t = a;
        a = b;
        b = t;
    }
    return a;
}

} // namespace mafx
