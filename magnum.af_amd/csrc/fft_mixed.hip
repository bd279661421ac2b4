// Axis kernels of the zero-padded demag convolution for lines of any length (factors up to 13), on
// the two-buffer LDS transform of fft_mixed.hpp, and two stages that keep a column in LDS from its
// forward transform to its inverse: the whole y stage of single-layer meshes (k_col) and the whole
// z stage of thick ones (k_zcol).  Spectrum layout and conventions as in fft.hip.
//
// All of them are sized per mesh: the tile shrinks until the launch has several work-groups per CU
// (or is one line per group), and the group has about one lane per eight tile elements.
//
// What bounds them: at small meshes the chain of latencies of a pass (load, two or three stages,
// store); at large ones the index and butterfly arithmetic (about 100 instructions per point and
// pass at radices 11 and 10).  Measured against the in-place kernels, us per launch:
//   700 x 330 x 3 FP32: x 67 -> 25 and 62 -> 23, y 102 -> 28 and 111 -> 29
//   100 x 25 x 1 FP64: x 15 -> 7 and 12 -> 6; y, product, y 12 + 4 + 17 -> 7 (k_col)
//   105 x 75 x 20 FP64: x 18 -> 15 and 16 -> 11, y 25 -> 13 and 34 -> 11; z, product, z
//   30 + 19 + 30 -> 32 (k_zcol)
#include <algorithm>
#include <functional>
#include <map>
#include <mutex>

#include "fft_kernels.hpp"
#include "fft_mixed.hpp"
#include "mafx_internal.hpp"

namespace mafx {

namespace {

// The schedule with the fewest stages and, among those, the smallest largest radix.  Powers of two
// keep the radix-8 schedule of FftPlan, whose results the compile-time shaped kernels share.
void mix_plan(int L, std::vector<int>& best) {
    best.clear();
    std::vector<int> cur;
    if (L == 1 || (L & (L - 1)) == 0) {
        for (int r : {8, 4, 2})
            while (L % r == 0) best.push_back(r), L /= r;
        return;
    }
    static const int radices[] = {16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    std::function<void(int, int)> go = [&](int n, int limit) {
        if (n == 1) {
            if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && cur[0] < best[0])) best = cur;
            return;
        }
        if (cur.size() >= static_cast<size_t>(kMixStages) || (!best.empty() && cur.size() >= best.size())) return;
        for (int r : radices)
            if (r <= limit && n % r == 0) {
                cur.push_back(r);
                go(n / r, r);
                cur.pop_back();
            }
    };
    go(L, 16);
}

const MixDesc& mix_desc(int L) {
    static std::mutex mu;
    static std::map<int, MixDesc> made; // one small entry per length ever used
    std::lock_guard<std::mutex> lk(mu);
    auto it = made.find(L);
    if (it != made.end()) return it->second;
    MixDesc d{};
    std::vector<int> r;
    mix_plan(L, r);
    d.L = L;
    if (r.size() <= static_cast<size_t>(kMixStages)) {
        int ns = 1;
        for (int R : r) {
            d.radix[d.nstages] = R;
            d.ns[d.nstages] = make_fastdiv(static_cast<uint32_t>(ns));
            ns *= R;
            d.twstep[d.nstages++] = L / ns;
        }
    }
    return made.emplace(L, d).first->second;
}

// The atomistic dipole field takes the kernels of this file where they give the sums of the in-place
// ones to the last bit: powers of two, up to 512 for the y column.  An LBFGS run on a spin lattice
// starts with line searches of some twenty evaluations whose steps turn spins by many radians; they
// take a last-bit difference of the field to percents of m within three iterations (a micromagnetic
// film's stay at 1e-15), so these runs are kept reproducible against earlier results.
bool reproducible(const mafx_ctx* ctx, int L) { return !ctx->atom_dipole || (L & (L - 1)) == 0; }

// Whether the schedule covers the length (a length of 1 needs no stage).
bool scheduled(const MixDesc& d) { return d.L == 1 || d.nstages > 0; }

template <class C> size_t mix_lds(int L, int lines, bool second = true) { return mix_lds_bytes(sizeof(C), L, lines, second); }

// Groups a launch should have before its tiles may grow: three per CU
int64_t mix_fill(const mafx_ctx* ctx) { return 3 * static_cast<int64_t>(ctx->num_cus); }

template <class C>
__device__ __forceinline__ void stage_twiddles(int M, const C* __restrict__ twh, const C* __restrict__ twL, C* tws, C* twl) {
    for (int t = threadIdx.x; t <= M; t += blockDim.x) {
        if (t < M) tws[t] = twh[t];
        twl[t] = twL[t];
    }
}

// Rows (c, z, y) of real input -> x half spectrum, W rows per group (k_fft_x_fwd's operation).
template <class C>
__global__ void __launch_bounds__(512)
    k_mix_x_fwd(const double* __restrict__ in, const double* __restrict__ ms, double scale, int Xi, int64_t Yi,
                int64_t Zi, FastDiv Yr, FastDiv Zr, int rows, FastDiv Wd, MixDesc d, FastDiv Md,
                const C* __restrict__ twh, const C* __restrict__ twL, C* __restrict__ out, int64_t hxs, int64_t n1,
                int64_t n2o) {
    using T = typename real_of<C>::type;
    extern __shared__ unsigned char smem_raw[];
    const int M = d.L, W = static_cast<int>(Wd.d), row0 = static_cast<int>(blockIdx.x) * W;
    C *A = reinterpret_cast<C*>(smem_raw), *B = A + lds_padded(M * W), *tws = B + lds_padded(M * W), *twl = tws + M;
    stage_twiddles(M, twh, twL, tws, twl);
    for (int e = threadIdx.x; e < M * W; e += blockDim.x) {
        const int w = static_cast<int>(fdiv(e, Md)), n = e - w * M, r = row0 + w;
        T re = 0, im = 0;
        if (r < rows) {
            const uint32_t zc = fdiv(r, Yr), y = r - zc * Yr.d, c = fdiv(zc, Zr), z = zc - c * Zr.d;
            const int64_t cell = (z * Yi + y) * Xi;
            const double* src = in + c * Zi * Yi * Xi + cell;
            const int t0 = 2 * n, t1 = t0 + 1;
            if (ms) {
                if (t0 < Xi) re = static_cast<T>(src[t0] * scale * ms[cell + t0]);
                if (t1 < Xi) im = static_cast<T>(src[t1] * scale * ms[cell + t1]);
            } else {
                if (t0 < Xi) re = static_cast<T>(src[t0] * scale);
                if (t1 < Xi) im = static_cast<T>(src[t1] * scale);
            }
        }
        A[lds_pad(n * W + w)] = C{re, im};
    }
    __syncthreads();
    const C* Z = mix_fft<C, false>(A, B, d, W, Wd, tws);
    const T half = static_cast<T>(0.5);
    const int64_t n1T = kTile * n1;
    const int ntile = (M + kTile) / kTile;
    // e = (kt W + w) 4 + kk: column k = 4 kt + kk of row w
    for (int e = threadIdx.x; e < ntile * W * kTile; e += blockDim.x) {
        const int kk = e & (kTile - 1), q = e >> 2, kt = static_cast<int>(fdiv(q, Wd)), w = q - kt * W;
        const int k = kt * kTile + kk, r = row0 + w;
        if (k > M || r >= rows) continue;
        const uint32_t zc = fdiv(r, Yr), y = r - zc * Yr.d, c = fdiv(zc, Zr), z = zc - c * Zr.d;
        const C Zk = Z[lds_pad((k == M ? 0 : k) * W + w)];
        const C Zm = Z[lds_pad((k == 0 ? 0 : M - k) * W + w)];
        const C E{half * (Zk.x + Zm.x), half * (Zk.y - Zm.y)};
        const C O{half * (Zk.y + Zm.y), -half * (Zk.x - Zm.x)};
        out[(c * n2o + z) * n1 * hxs + kTile * static_cast<int64_t>(y) + tcol(k, n1T)] = cadd(E, cmul(twl[k], O));
    }
}

// x half spectrum -> real rows, cropped and scaled (k_fft_x_inv's operation).
template <class C, class T>
__global__ void __launch_bounds__(512)
    k_mix_x_inv(const C* __restrict__ spec, int64_t hxs, int64_t n1, int64_t n2s, FastDiv Yr, FastDiv Zr, int rows,
                FastDiv Wd, MixDesc d, FastDiv Mhd, const C* __restrict__ twh, const C* __restrict__ twL,
                T* __restrict__ out, int Xo, double hscale) {
    extern __shared__ unsigned char smem_raw[];
    const int M = d.L, W = static_cast<int>(Wd.d), row0 = static_cast<int>(blockIdx.x) * W;
    C *A = reinterpret_cast<C*>(smem_raw), *B = A + lds_padded(M * W), *tws = B + lds_padded(M * W);
    for (int t = threadIdx.x; t < M; t += blockDim.x) tws[t] = twh[t];
    const int64_t n1T = kTile * n1;
    const int ntile = (M + kTile - 1) / kTile;
    for (int e = threadIdx.x; e < ntile * W * kTile; e += blockDim.x) {
        const int kk = e & (kTile - 1), q = e >> 2, kt = static_cast<int>(fdiv(q, Wd)), w = q - kt * W;
        const int k = kt * kTile + kk, r = row0 + w;
        if (k >= M) continue;
        C v{0, 0};
        if (r < rows) {
            const uint32_t zc = fdiv(r, Yr), y = r - zc * Yr.d, c = fdiv(zc, Zr), z = zc - c * Zr.d;
            const C* s = spec + (c * n2s + z) * n1 * hxs + kTile * static_cast<int64_t>(y);
            v = c2r_combine(s[tcol(k, n1T)], s[tcol(M - k, n1T)], twL[k]);
        }
        A[lds_pad(k * W + w)] = v;
    }
    __syncthreads();
    const C* Z = mix_fft<C, true>(A, B, d, W, Wd, tws);
    const int Mh = static_cast<int>(Mhd.d);
    for (int e = threadIdx.x; e < Mh * W; e += blockDim.x) {
        const int w = static_cast<int>(fdiv(e, Mhd)), n = e - w * Mh, r = row0 + w;
        if (r >= rows) continue;
        // row r of the output is at r Xo: (c, z, y) run as in memory
        T* o = out + static_cast<int64_t>(r) * Xo + 2 * n;
        const C v = Z[lds_pad(n * W + w)];
        o[0] = static_cast<T>(static_cast<double>(v.x) * hscale);
        if (2 * n + 1 < Xo) o[1] = static_cast<T>(static_cast<double>(v.y) * hscale);
    }
}

// Both halves of the zero-padded y transform of W columns (k_fft_y_fwd2's operation): line w holds
// x[n] (outputs X[2k]), line W + w holds x[n] w_L^n (outputs X[2k+1]).
template <class C>
__global__ void __launch_bounds__(512)
    k_mix_y_fwd(C* __restrict__ data, int64_t plane, int hx, FastDiv Wd, FastDiv W2d, MixDesc d,
                const C* __restrict__ twh, const C* __restrict__ twL, int64_t n1T) {
    extern __shared__ unsigned char smem_raw[];
    const int M = d.L, W = static_cast<int>(Wd.d), W2 = 2 * W;
    C *A = reinterpret_cast<C*>(smem_raw), *B = A + lds_padded(M * W2), *tws = B + lds_padded(M * W2);
    for (int t = threadIdx.x; t < M; t += blockDim.x) tws[t] = twh[t];
    const uint3 blk = swizzled_block();
    const int kx0 = static_cast<int>(blk.x) * W;
    C* base = data + static_cast<int64_t>(blk.y) * plane;
    for (int e = threadIdx.x; e < M * W; e += blockDim.x) {
        const int n = static_cast<int>(fdiv(e, Wd)), w = e - n * W;
        const C v = kx0 + w < hx ? base[kTile * n + tcol(kx0 + w, n1T)] : C{0, 0}, t = twL[n];
        A[lds_pad(n * W2 + w)] = v;
        A[lds_pad(n * W2 + W + w)] = cmul(v, t);
    }
    __syncthreads();
    const C* X = mix_fft<C, false>(A, B, d, W2, W2d, tws);
    for (int e = threadIdx.x; e < M * W2; e += blockDim.x) {
        const int ky = static_cast<int>(fdiv(e, Wd)), w = e - ky * W; // ky = 2 k + odd
        if (kx0 + w < hx) base[kTile * ky + tcol(kx0 + w, n1T)] = X[lds_pad((ky >> 1) * W2 + (ky & 1) * W + w)];
    }
}

// Inverse counterpart: x[n] = IFFT_M(X_even)[n] + w_L^-n IFFT_M(X_odd)[n], n < M.
template <class C>
__global__ void __launch_bounds__(512)
    k_mix_y_inv(C* __restrict__ data, int64_t plane, int hx, FastDiv Wd, FastDiv W2d, MixDesc d,
                const C* __restrict__ twh, const C* __restrict__ twL, int64_t n1T) {
    extern __shared__ unsigned char smem_raw[];
    const int M = d.L, W = static_cast<int>(Wd.d), W2 = 2 * W;
    C *A = reinterpret_cast<C*>(smem_raw), *B = A + lds_padded(M * W2), *tws = B + lds_padded(M * W2), *twl = tws + M;
    stage_twiddles(M, twh, twL, tws, twl);
    const uint3 blk = swizzled_block();
    const int kx0 = static_cast<int>(blk.x) * W;
    C* base = data + static_cast<int64_t>(blk.y) * plane;
    for (int e = threadIdx.x; e < M * W2; e += blockDim.x) {
        const int ky = static_cast<int>(fdiv(e, Wd)), w = e - ky * W;
        A[lds_pad((ky >> 1) * W2 + (ky & 1) * W + w)] =
            kx0 + w < hx ? base[kTile * ky + tcol(kx0 + w, n1T)] : C{0, 0};
    }
    __syncthreads();
    const C* x = mix_fft<C, true>(A, B, d, W2, W2d, tws);
    for (int e = threadIdx.x; e < M * W; e += blockDim.x) {
        const int n = static_cast<int>(fdiv(e, Wd)), w = e - n * W;
        if (kx0 + w < hx)
            base[kTile * n + tcol(kx0 + w, n1T)] =
                cadd(x[lds_pad(n * W2 + w)], cmul(conj_if(twl[n], true), x[lds_pad(n * W2 + W + w)]));
    }
}

// The tensor at one k-point and its product with (X0, X1, X2), in the three stored forms: FULL the
// complex spectrum [6][n2][plane]; SYM the real symmetric quarter (fft.hip: signs sy, sz of the
// mirrored ky, kz); SYMRES the quarter plus the FP16 residual of the whole spectrum.
enum { kFull = 0, kSym = 1, kSymRes = 2 };
template <class C> struct TensorArg {
    const void* t;
    TensorRes res;
    int n1, n2, n1h, n2h; // rows, planes and their mirror extents
    int64_t hxs;
};
template <class C, int FORM>
__device__ __forceinline__ void tensor_product(const TensorArg<C>& a, int kx, int ky, int kz, C& X0, C& X1, C& X2) {
    const int64_t plane = static_cast<int64_t>(a.n1) * a.hxs, K = a.n2 * plane;
    const int64_t i = kz * plane + tcol(kx, kTile * static_cast<int64_t>(a.n1)) + kTile * ky;
    const C x0 = X0, x1 = X1, x2 = X2;
    if constexpr (FORM == kFull) {
        const C* t = static_cast<const C*>(a.t) + i;
        const C xx = t[0], xy = t[K], xz = t[2 * K], yy = t[3 * K], yz = t[4 * K], zz = t[5 * K];
        X0 = cadd(cadd(cmul(xx, x0), cmul(xy, x1)), cmul(xz, x2));
        X1 = cadd(cadd(cmul(xy, x0), cmul(yy, x1)), cmul(yz, x2));
        X2 = cadd(cadd(cmul(xz, x0), cmul(yz, x1)), cmul(zz, x2));
    } else {
        const bool my = ky >= a.n1h, mz = kz >= a.n2h;
        const int kys = my ? a.n1 - ky : ky, kzs = mz ? a.n2 - kz : kz;
        const float sy = my ? -1.0f : 1.0f, sz = mz ? -1.0f : 1.0f;
        const int64_t Q = static_cast<int64_t>(a.n1h) * a.hxs, tc = a.n2h * Q;
        const float* t = static_cast<const float*>(a.t) + kzs * Q + tcol(kx, kTile * a.n1h) + kTile * kys;
        const float s[6] = {t[0], sy * t[tc], sz * t[2 * tc], t[3 * tc], sy * sz * t[4 * tc], t[5 * tc]};
        if constexpr (FORM == kSymRes) {
            C T[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                const float2 r = __half22float2(a.res.r[c * K + i]);
                T[c] = C{s[c] + r.x * a.res.inv[c], r.y * a.res.inv[c]};
            }
            X0 = cadd(cadd(cmul(T[0], x0), cmul(T[1], x1)), cmul(T[2], x2));
            X1 = cadd(cadd(cmul(T[1], x0), cmul(T[3], x1)), cmul(T[4], x2));
            X2 = cadd(cadd(cmul(T[2], x0), cmul(T[4], x1)), cmul(T[5], x2));
        } else {
            X0 = C{s[0] * x0.x + s[1] * x1.x + s[2] * x2.x, s[0] * x0.y + s[1] * x1.y + s[2] * x2.y};
            X1 = C{s[1] * x0.x + s[3] * x1.x + s[4] * x2.x, s[1] * x0.y + s[3] * x1.y + s[4] * x2.y};
            X2 = C{s[2] * x0.x + s[4] * x1.x + s[5] * x2.x, s[2] * x0.y + s[4] * x1.y + s[5] * x2.y};
        }
    }
}

// The whole y stage of a single-layer mesh: zero-padded forward y transform, tensor product and
// cropped inverse of W columns and the three components without leaving LDS, in place on rows
// y < ny.  One launch and one pass over half the spectrum instead of three over all of it.  The even
// and the odd ky (the split of k_mix_y_fwd) are transformed together (NH = 2) or, where six lines per
// column do not fit a useful tile, one after the other (NH = 1): the first half's outputs then wait
// in registers, at most kColAcc per lane (col_tile).
template <class C, int FORM, int NH>
__global__ void __launch_bounds__(512)
    k_col(C* __restrict__ spec, int64_t plane, TensorArg<C> ta, int hx, FastDiv Wd, FastDiv lined, MixDesc d, FastDiv Md,
          const C* __restrict__ twh, const C* __restrict__ twL) {
    extern __shared__ unsigned char smem_raw[];
    const int M = d.L, W = static_cast<int>(Wd.d), NL = 3 * NH * W, MW = M * W;
    C *A = reinterpret_cast<C*>(smem_raw), *B = A + lds_padded(M * NL), *tws = B + lds_padded(M * NL), *twl = tws + M;
    stage_twiddles(M, twh, twL, tws, twl);
    const int kx0 = static_cast<int>(xcd_swizzle(blockIdx.x, gridDim.x)) * W;
    const int64_t n1T = kTile * static_cast<int64_t>(ta.n1);
    C acc[NH == 1 ? kColAcc : 1];
#pragma unroll 1
    for (int h0 = 0; h0 < 2; h0 += NH) {
        // e = (c M + y) W + w
        for (int e = threadIdx.x; e < 3 * MW; e += blockDim.x) {
            const int r = static_cast<int>(fdiv(e, Wd)), w = e - r * W, c = static_cast<int>(fdiv(r, Md)), y = r - c * M;
            const C v = kx0 + w < hx ? spec[c * plane + tcol(kx0 + w, n1T) + kTile * y] : C{0, 0};
            if constexpr (NH == 2) {
                A[lds_pad(y * NL + 2 * c * W + w)] = v;
                A[lds_pad(y * NL + (2 * c + 1) * W + w)] = cmul(v, twL[y]);
            } else {
                A[lds_pad(y * NL + c * W + w)] = h0 ? cmul(v, twL[y]) : v;
            }
        }
        __syncthreads();
        C* X = mix_fft<C, false>(A, B, d, NL, lined, tws);
        // e = (k NH + h) W + w: ky = 2 k + h0 + h
        for (int e = threadIdx.x; e < MW * NH; e += blockDim.x) {
            const int r = static_cast<int>(fdiv(e, Wd)), w = e - r * W, k = NH == 2 ? r >> 1 : r, h = NH == 2 ? r & 1 : 0;
            if (kx0 + w >= hx) continue;
            const int i0 = lds_pad(k * NL + h * W + w), i1 = lds_pad(k * NL + (NH + h) * W + w),
                      i2 = lds_pad(k * NL + (2 * NH + h) * W + w);
            C x0 = X[i0], x1 = X[i1], x2 = X[i2];
            tensor_product<C, FORM>(ta, kx0 + w, 2 * k + h0 + h, 0, x0, x1, x2);
            X[i0] = x0;
            X[i1] = x1;
            X[i2] = x2;
        }
        __syncthreads();
        const C* x = mix_fft<C, true>(X, X == A ? B : A, d, NL, lined, tws);
        if constexpr (NH == 2) {
            for (int e = threadIdx.x; e < 3 * MW; e += blockDim.x) {
                const int r = static_cast<int>(fdiv(e, Wd)), w = e - r * W, c = static_cast<int>(fdiv(r, Md)), y = r - c * M;
                if (kx0 + w < hx)
                    spec[c * plane + tcol(kx0 + w, n1T) + kTile * y] =
                        cadd(x[lds_pad(y * NL + 2 * c * W + w)],
                             cmul(conj_if(twl[y], true), x[lds_pad(y * NL + (2 * c + 1) * W + w)]));
            }
        } else {
            // a lane's i-th element is the same in both halves; 3 M W <= kColAcc blockDim
#pragma unroll
            for (int i = 0; i < kColAcc; ++i) {
                const int e = threadIdx.x + i * blockDim.x;
                if (e < 3 * MW) {
                    const int r = static_cast<int>(fdiv(e, Wd)), w = e - r * W, c = static_cast<int>(fdiv(r, Md)), y = r - c * M;
                    const C v = x[lds_pad(y * NL + c * W + w)];
                    if (h0 == 0)
                        acc[i] = v;
                    else if (kx0 + w < hx)
                        spec[c * plane + tcol(kx0 + w, n1T) + kTile * y] = cadd(acc[i], cmul(conj_if(twl[y], true), v));
                }
            }
            __syncthreads(); // the next half's inputs overwrite the buffers
        }
    }
}

// k_col for power-of-two ny = 2^LOGM on the compile-time shaped in-place stages of fft_device.hpp:
// 2^LOGE complex values (W2 = 2 W lines: the even and odd halves of W columns) and 2^LOGE / 8 lanes
// per component, so that every lane owns one radix-8 butterfly of a stage; the three components are
// transformed side by side by the group's three thirds, and meet in the tensor product.  Bound by
// the tensor's bytes in FP64 (51 of 76 MB at 1024 x 256 and 512 x 512): 20 us against 12 + 17 + 11
// for the three passes at 1024 x 256, 29 against 12 + 17 + 11 at 512 x 512, where a column's two lines
// fill the 16 KiB and each group reads 16 of every 64 bytes.  Its last forward and inverse stages are
// written like those of k_fft_y_fwd_ct and k_fft_y_inv_ct, so the sums stay theirs to the last bit up
// to ny = 512.
template <class C, int FORM, int LOGM, int LOGE>
__global__ void __launch_bounds__(3 << (LOGE - 3))
    k_col_ct(C* __restrict__ spec, int64_t plane, TensorArg<C> ta, int hx, const C* __restrict__ twh,
             const C* __restrict__ twL) {
    constexpr int M = 1 << LOGM, LOGW2 = LOGE - LOGM, W2 = 1 << LOGW2, LOGW = LOGW2 - 1, W = W2 / 2;
    constexpr int BSC = 1 << (LOGE - 3), BS = 3 * BSC, IT = 4; // M W / BSC inputs per lane
    constexpr int NST = ct_nstages(LOGM);
    using SL = CtStage<LOGM, LOGW2, NST - 1>;
    constexpr int NBL = SL::NB / BSC, H = SL::R / 2; // last-stage butterflies per lane
    static_assert(LOGW >= 0 && W <= kTile && BSC % 64 == 0 && W2 <= 64 && SL::NB % BSC == 0 && SL::R >= 2, "tile shape");
    extern __shared__ unsigned char smem_raw[];
    constexpr int REG = lds_padded(1 << LOGE);
    C *buf = reinterpret_cast<C*>(smem_raw), *tws = buf + 3 * REG;
    const int tid = static_cast<int>(threadIdx.x), c = tid / BSC, lt = tid % BSC;
    for (int t = tid; t < M; t += BS) tws[t] = twh[t];
    const int kx0 = static_cast<int>(xcd_swizzle(blockIdx.x, gridDim.x)) * W;
    const int64_t n1T = kTile * static_cast<int64_t>(ta.n1);
    C* cb = buf + c * REG;
    C* base = spec + c * plane;
    C v[IT], t[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int g = lt + i * BSC, y = g >> LOGW, w = g & (W - 1);
        v[i] = kx0 + w < hx ? base[tcol(kx0 + w, n1T) + kTile * y] : C{0, 0};
        t[i] = twL[y];
    }
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int g = lt + i * BSC, y = g >> LOGW, w = g & (W - 1);
        cb[lds_pad((y << LOGW2) + w)] = v[i];
        cb[lds_pad((y << LOGW2) + W + w)] = cmul(v[i], t[i]);
    }
    __syncthreads();
    ct_fft<C, LOGM, LOGW2, BSC, false, 0, NST - 1>(cb, tws, lt);
    {
        // the last stage, as k_fft_y_fwd_ct writes it to memory (the same bits)
        C u[NBL][SL::R];
#pragma unroll
        for (int i = 0; i < NBL; ++i)
#pragma unroll
            for (int r = 0; r < SL::R; ++r) u[i][r] = cb[lds_pad(lt + i * BSC + r * SL::NB)];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NBL; ++i) {
            const int b = lt + i * BSC, l = b & (W2 - 1);
            SL::template bfly<C, false>(u[i], b, tws);
            if (kx0 + (l & (W - 1)) < hx)
#pragma unroll
                for (int r = 0; r < SL::R; ++r) cb[lds_pad((SL::opos(b, r) << LOGW2) + l)] = u[i][r];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 3; ++i) { // 8 / 3 k-points per lane
        const int e = tid + i * BS, k = e >> LOGW2, l = e & (W2 - 1), odd = l >> LOGW, w = l & (W - 1);
        if (e < (1 << LOGE) && kx0 + w < hx) {
            C* q = buf + lds_pad(e);
            C x0 = q[0], x1 = q[REG], x2 = q[2 * REG];
            tensor_product<C, FORM>(ta, kx0 + w, 2 * k + odd, 0, x0, x1, x2);
            q[0] = x0;
            q[REG] = x1;
            q[2 * REG] = x2;
        }
    }
    __syncthreads();
    ct_fft<C, LOGM, LOGW2, BSC, true, 0, NST - 1>(cb, tws, lt);
    // the last stage leaves IFFT_M(X_even)[n] and IFFT_M(X_odd)[n] of column w in lanes b and b ^ W
    // of one wave, which trade half of their outputs (k_fft_y_inv_ct)
#pragma unroll
    for (int i = 0; i < NBL; ++i) {
        const int b = lt + i * BSC, j = b >> LOGW2, l = b & (W2 - 1), w = l & (W - 1), odd = l >> LOGW;
        C u[SL::R];
#pragma unroll
        for (int r = 0; r < SL::R; ++r) u[r] = cb[lds_pad(b + r * SL::NB)];
        SL::template bfly<C, true>(u, b, tws);
        const bool ok = kx0 + w < hx;
        C* dst = base + tcol(kx0 + w, n1T);
#pragma unroll
        for (int q = 0; q < H; ++q) {
            const C give = odd ? u[q] : u[q + H];
            const C recv{__shfl_xor(give.x, W, 64), __shfl_xor(give.y, W, 64)};
            const int n = j + (odd ? q + H : q) * SL::NS;
            const C e = odd ? recv : u[q], o = odd ? u[q + H] : recv;
            if (ok) dst[kTile * n] = cadd(e, cmul(conj_if(twL[n], true), o));
        }
    }
}

// The whole z stage of a mesh of more than eight layers: forward transform of the nz non-zero planes
// (length 2 nz), tensor product per kz, inverse kept for z < nz, for W neighbouring positions of the
// plane and the three components in LDS.  Spectrum planes [3][nz][plane], in place.
template <class C, int FORM>
__global__ void __launch_bounds__(512)
    k_zcol(C* __restrict__ spec, int64_t plane, TensorArg<C> ta, int nz, int npos, FastDiv Wd, FastDiv lined, MixDesc d,
           FastDiv nzd, FastDiv n1Td, const C* __restrict__ tw) {
    extern __shared__ unsigned char smem_raw[];
    const int L = d.L, W = static_cast<int>(Wd.d), NL = 3 * W;
    C *A = reinterpret_cast<C*>(smem_raw), *B = A + lds_padded(L * NL), *tws = B + lds_padded(L * NL);
    for (int t = threadIdx.x; t < L; t += blockDim.x) tws[t] = tw[t];
    const int p0 = static_cast<int>(blockIdx.x) * W;
    // e = (c nz + z) W + w
    for (int e = threadIdx.x; e < nz * NL; e += blockDim.x) {
        const int r = static_cast<int>(fdiv(e, Wd)), w = e - r * W, c = static_cast<int>(fdiv(r, nzd)), z = r - c * nz;
        const C v = p0 + w < npos ? spec[r * plane + p0 + w] : C{0, 0};
        A[lds_pad(z * NL + c * W + w)] = v;
        A[lds_pad((z + nz) * NL + c * W + w)] = C{0, 0};
    }
    __syncthreads();
    C* X = mix_fft<C, false>(A, B, d, NL, lined, tws);
    for (int e = threadIdx.x; e < L * W; e += blockDim.x) {
        const int kz = static_cast<int>(fdiv(e, Wd)), w = e - kz * W, p = p0 + w;
        if (p >= npos) continue;
        const int kt = static_cast<int>(fdiv(p, n1Td)), r = p - kt * static_cast<int>(n1Td.d);
        const int i0 = lds_pad(kz * NL + w), i1 = lds_pad(kz * NL + W + w), i2 = lds_pad(kz * NL + 2 * W + w);
        C x0 = X[i0], x1 = X[i1], x2 = X[i2];
        tensor_product<C, FORM>(ta, kt * kTile + (r & (kTile - 1)), r >> 2, kz, x0, x1, x2);
        X[i0] = x0;
        X[i1] = x1;
        X[i2] = x2;
    }
    __syncthreads();
    const C* x = mix_fft<C, true>(X, X == A ? B : A, d, NL, lined, tws);
    for (int e = threadIdx.x; e < nz * NL; e += blockDim.x) {
        const int r = static_cast<int>(fdiv(e, Wd)), w = e - r * W, c = static_cast<int>(fdiv(r, nzd)), z = r - c * nz;
        if (p0 + w < npos) spec[r * plane + p0 + w] = x[lds_pad(z * NL + c * W + w)];
    }
}

// Lines per group along x: whole column tiles' worth of rows (4) where the mesh has enough of them
template <class C> int x_rows(const mafx_ctx* ctx, int M, int64_t rows) {
    for (int W : {8, 4, 2, 1})
        if (mix_lds<C>(M, W) <= (W > 1 ? size_t{56} * 1024 : kLdsMax) && (W == 1 || rows / W >= mix_fill(ctx))) return W;
    return 0;
}

} // namespace

template <class C>
bool mix_x_forward(mafx_ctx* ctx, const double* in, const double* ms, double scale, int64_t Xi, int64_t Yi, int64_t Zi,
                   int ncomp, int64_t Yr, int64_t Zr, C* out, int64_t n2o) {
    const MixDesc& d = mix_desc(ctx->pxh.L);
    const int M = d.L;
    const int64_t rows = static_cast<int64_t>(ncomp) * Zr * Yr;
    const int W = scheduled(d) && reproducible(ctx, M) ? x_rows<C>(ctx, M, rows) : 0;
    if (W == 0) return false;
    require(rows * (M + 1) < (int64_t{1} << 31) && Xi < (int64_t{1} << 30), "x transform: too many rows");
    ProfScope ps(ctx, nm("fft_x_fwd_f32", "fft_x_fwd_f64", sizeof(C)),
                 static_cast<double>(rows) * (Xi * 8.0 + ctx->hx * sizeof(C)));
    const size_t lds = mix_lds<C>(M, W);
    allow_lds(reinterpret_cast<const void*>(k_mix_x_fwd<C>), lds);
    hipLaunchKernelGGL(k_mix_x_fwd<C>, dim3(static_cast<unsigned>((rows + W - 1) / W)), dim3(mix_block(M * W)), lds,
                       ctx->stream, in, ms, scale, static_cast<int>(Xi), Yi, Zi, make_fastdiv(static_cast<uint32_t>(Yr)),
                       make_fastdiv(static_cast<uint32_t>(Zr)), static_cast<int>(rows), make_fastdiv(W), d,
                       make_fastdiv(M), tw_of<C>(ctx->pxh), tw_of<C>(ctx->px), out, ctx->hxs, ctx->n1, n2o);
    MAFX_HIP(hipGetLastError());
    return true;
}

template <class C, class T> bool mix_x_inverse(mafx_ctx* ctx, const C* spec, int64_t n2s, T* out, double hscale) {
    const MixDesc& d = mix_desc(ctx->pxh.L);
    const int M = d.L;
    const mafx_mesh& g = ctx->mesh;
    const int64_t rows = 3 * g.nz * g.ny;
    const int W = scheduled(d) && reproducible(ctx, M) ? x_rows<C>(ctx, M, rows) : 0;
    if (W == 0) return false;
    require(rows * (M + 1) < (int64_t{1} << 31), "x transform: too many rows");
    ProfScope ps(ctx, nm("fft_x_inv_f32", "fft_x_inv_f64", sizeof(C)),
                 static_cast<double>(rows) * (ctx->hx * sizeof(C) + g.nx * sizeof(T)));
    const size_t lds = mix_lds<C>(M, W);
    allow_lds(reinterpret_cast<const void*>(k_mix_x_inv<C, T>), lds);
    hipLaunchKernelGGL((k_mix_x_inv<C, T>), dim3(static_cast<unsigned>((rows + W - 1) / W)), dim3(mix_block(M * W)), lds,
                       ctx->stream, spec, ctx->hxs, ctx->n1, n2s, make_fastdiv(static_cast<uint32_t>(g.ny)),
                       make_fastdiv(static_cast<uint32_t>(g.nz)), static_cast<int>(rows), make_fastdiv(W), d,
                       make_fastdiv(static_cast<uint32_t>((g.nx + 1) / 2)), tw_of<C>(ctx->pxh), tw_of<C>(ctx->px), out,
                       static_cast<int>(g.nx), hscale);
    MAFX_HIP(hipGetLastError());
    return true;
}

template <class C> bool mix_y_split(mafx_ctx* ctx, C* data, int nplanes, bool inv) {
    const MixDesc& d = mix_desc(ctx->pyh.L);
    const int M = d.L;
    if (!scheduled(d) || !reproducible(ctx, M) || nplanes > 65535) return false;
    const int hx = static_cast<int>(ctx->hx);
    int W = 0;
    for (int w : {4, 2, 1})
        if (mix_lds<C>(M, 2 * w) <= (w > 1 ? size_t{80} * 1024 : kLdsMax) &&
            (w == 1 || static_cast<int64_t>((hx + w - 1) / w) * nplanes >= mix_fill(ctx))) {
            W = w;
            break;
        }
    if (W == 0) return false;
    ProfScope ps(ctx, inv ? nm("fft_y_inv_f32", "fft_y_inv_f64", sizeof(C)) : nm("fft_y_fwd_f32", "fft_y_fwd_f64", sizeof(C)),
                 static_cast<double>(nplanes) * ctx->hx * (3.0 * M) * sizeof(C));
    const size_t lds = mix_lds<C>(M, 2 * W);
    auto fn = inv ? k_mix_y_inv<C> : k_mix_y_fwd<C>;
    allow_lds(reinterpret_cast<const void*>(fn), lds);
    hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>((hx + W - 1) / W), static_cast<unsigned>(nplanes)),
                       dim3(mix_block(2 * M * W)), lds, ctx->stream, data, ctx->n1 * ctx->hxs, hx, make_fastdiv(W),
                       make_fastdiv(2 * W), d, tw_of<C>(ctx->pyh), tw_of<C>(ctx->py), kTile * ctx->n1);
    MAFX_HIP(hipGetLastError());
    return true;
}

namespace {
template <class C> TensorArg<C> tensor_arg(const mafx_ctx* ctx, const C* full, const float* sym, const TensorRes* res) {
    TensorArg<C> a{};
    a.t = full ? static_cast<const void*>(full) : static_cast<const void*>(sym);
    if (res) a.res = *res;
    a.n1 = static_cast<int>(ctx->n1);
    a.n2 = static_cast<int>(ctx->n2);
    a.n1h = static_cast<int>(ctx->n1h);
    a.n2h = static_cast<int>(ctx->n2h);
    a.hxs = ctx->hxs;
    return a;
}
// algorithmic bytes of the tensor over n2 planes
template <class C> double tensor_bytes(const mafx_ctx* ctx, bool full, bool res) {
    const double K = static_cast<double>(ctx->n2 * ctx->n1 * ctx->hx);
    return full ? 6.0 * sizeof(C) * K
                : 6.0 * sizeof(float) * static_cast<double>(ctx->n2h * ctx->n1h * ctx->hx) + (res ? 6.0 * sizeof(__half2) * K : 0.0);
}
// Tile of k_col_ct for a power-of-two ny of 128..1024: 16 KiB per component (three groups per CU),
// or the two lines a column needs; smaller, down to one column, while the groups do not fill the chip.
template <class C, int FORM> bool col_ct_launch(mafx_ctx* ctx, C* spec, const TensorArg<C>& ta) {
    const int M = ctx->pyh.L, hx = static_cast<int>(ctx->hx);
    if (M < 128 || M > 1024 || (M & (M - 1)) != 0) return false;
    int logm = 0;
    while ((1 << logm) < M) ++logm;
    int loge = std::max(sizeof(C) == sizeof(float2) ? 11 : 10, logm + 1);
    const auto groups = [&](int le) {
        const int W = 1 << (le - logm - 1);
        return (hx + W - 1) / W;
    };
    loge = std::min(loge, logm + 3); // at most one column tile
    while (loge > std::max(9, logm + 1) && groups(loge) < mix_fill(ctx)) --loge;
    using KC = void (*)(C*, int64_t, TensorArg<C>, int, const C*, const C*);
    KC fn = nullptr;
    switch (100 * logm + loge) {
#define MAFX_COL(LM, LE) \
    case 100 * LM + LE: fn = k_col_ct<C, FORM, LM, LE>; break;
        MAFX_COL(7, 9)
        MAFX_COL(7, 10)
        MAFX_COL(8, 9)
        MAFX_COL(8, 10)
        MAFX_COL(8, 11)
        MAFX_COL(9, 10)
        MAFX_COL(9, 11)
        MAFX_COL(10, 11)
#undef MAFX_COL
    default: return false;
    }
    ProfScope ps(ctx, nm("ycol_mul_f32", "ycol_mul_f64", sizeof(C)),
                 6.0 * static_cast<double>(M) * ctx->hx * sizeof(C) + tensor_bytes<C>(ctx, FORM == kFull, FORM == kSymRes));
    const size_t lds = (3 * static_cast<size_t>(lds_padded(1 << loge)) + M) * sizeof(C);
    allow_lds(reinterpret_cast<const void*>(fn), lds);
    hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(groups(loge))), dim3(3u << (loge - 3)), lds, ctx->stream, spec,
                       ctx->nzs * ctx->n1 * ctx->hxs, ta, hx, tw_of<C>(ctx->pyh), tw_of<C>(ctx->py));
    MAFX_HIP(hipGetLastError());
    return true;
}
template <class C, int FORM> bool col_launch(mafx_ctx* ctx, C* spec, const TensorArg<C>& ta) {
    if (!reproducible(ctx, ctx->pyh.L) || (ctx->atom_dipole && ctx->pyh.L > 512)) return false;
    if (col_ct_launch<C, FORM>(ctx, spec, ta)) return true;
    const MixDesc& d = mix_desc(ctx->pyh.L);
    const int M = d.L, hx = static_cast<int>(ctx->hx);
    if (!scheduled(d)) return false;
    const ColTile t = col_tile(sizeof(C), M, hx, mix_fill(ctx));
    const int W = t.W, NH = t.NH, lines = 3 * NH * W;
    if (W == 0) return false;
    require(NH == 2 || 3 * M * W <= kColAcc * t.block, "y column: more outputs than its lanes keep");
    ProfScope ps(ctx, nm("ycol_mul_f32", "ycol_mul_f64", sizeof(C)),
                 6.0 * static_cast<double>(M) * ctx->hx * sizeof(C) + tensor_bytes<C>(ctx, FORM == kFull, FORM == kSymRes));
    const size_t lds = mix_lds<C>(M, lines);
    auto fn = NH == 2 ? k_col<C, FORM, 2> : k_col<C, FORM, 1>;
    allow_lds(reinterpret_cast<const void*>(fn), lds);
    hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>((hx + W - 1) / W)), dim3(t.block), lds, ctx->stream, spec,
                       ctx->nzs * ctx->n1 * ctx->hxs, ta, hx, make_fastdiv(W), make_fastdiv(lines), d,
                       make_fastdiv(M), tw_of<C>(ctx->pyh), tw_of<C>(ctx->py));
    MAFX_HIP(hipGetLastError());
    return true;
}
template <class C> int zcol_width(int nz) {
    for (int w : {16, 8, 4, 2, 1})
        if (mix_lds<C>(2 * nz, 3 * w, false) <= (w > 4 ? size_t{40} * 1024 : w > 1 ? size_t{80} * 1024 : kLdsMax)) return w;
    return 0;
}
template <class C, int FORM> void zcol_launch(mafx_ctx* ctx, C* spec, const TensorArg<C>& ta) {
    const int nz = static_cast<int>(ctx->mesh.nz), W = zcol_width<C>(nz);
    const MixDesc& d = mix_desc(ctx->pz.L);
    require(W > 0 && scheduled(d), "z stage: column exceeds the LDS budget");
    // whole column tiles hold every column kx < hx; the padding beyond them is never read
    const int64_t npos = (ctx->hx + kTile - 1) / kTile * kTile * ctx->n1;
    require(npos < (int64_t{1} << 31), "spectrum too large for the z stage");
    ProfScope ps(ctx, nm("zcol_mul_f32", "zcol_mul_f64", sizeof(C)),
                 static_cast<double>(ctx->n1 * ctx->hx) * 6.0 * nz * sizeof(C) +
                     tensor_bytes<C>(ctx, FORM == kFull, FORM == kSymRes));
    const size_t lds = mix_lds<C>(2 * nz, 3 * W, false);
    auto fn = k_zcol<C, FORM>;
    allow_lds(reinterpret_cast<const void*>(fn), lds);
    hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>((npos + W - 1) / W)), dim3(mix_block(6 * nz * W)), lds, ctx->stream,
                       spec, ctx->n1 * ctx->hxs, ta, nz, static_cast<int>(npos), make_fastdiv(W), make_fastdiv(3 * W), d,
                       make_fastdiv(nz), make_fastdiv(static_cast<uint32_t>(kTile * ctx->n1)), tw_of<C>(ctx->pz));
    MAFX_HIP(hipGetLastError());
}
} // namespace

bool y_column(mafx_ctx* ctx, double2* spec, const double2* t) {
    return col_launch<double2, kFull>(ctx, spec, tensor_arg<double2>(ctx, t, nullptr, nullptr));
}
bool y_column(mafx_ctx* ctx, float2* spec, const float* t, const TensorRes* res) {
    const auto ta = tensor_arg<float2>(ctx, nullptr, t, res);
    return res ? col_launch<float2, kSymRes>(ctx, spec, ta) : col_launch<float2, kSym>(ctx, spec, ta);
}
bool z_column_fits(const mafx_ctx* ctx, bool f64) {
    const int64_t nz = ctx->mesh.nz;
    return nz < (int64_t{1} << 20) && !ctx->atom_dipole && scheduled(mix_desc(ctx->pz.L)) &&
           (f64 ? zcol_width<double2>(static_cast<int>(nz)) : zcol_width<float2>(static_cast<int>(nz))) > 0;
}
void z_column(mafx_ctx* ctx, double2* spec, const double2* t) {
    zcol_launch<double2, kFull>(ctx, spec, tensor_arg<double2>(ctx, t, nullptr, nullptr));
}
void z_column(mafx_ctx* ctx, float2* spec, const float* t, const TensorRes* res) {
    const auto ta = tensor_arg<float2>(ctx, nullptr, t, res);
    if (res)
        zcol_launch<float2, kSymRes>(ctx, spec, ta);
    else
        zcol_launch<float2, kSym>(ctx, spec, ta);
}

template bool mix_x_forward<double2>(mafx_ctx*, const double*, const double*, double, int64_t, int64_t, int64_t, int,
                                     int64_t, int64_t, double2*, int64_t);
template bool mix_x_forward<float2>(mafx_ctx*, const double*, const double*, double, int64_t, int64_t, int64_t, int,
                                    int64_t, int64_t, float2*, int64_t);
template bool mix_x_inverse<double2, double>(mafx_ctx*, const double2*, int64_t, double*, double);
template bool mix_x_inverse<float2, float>(mafx_ctx*, const float2*, int64_t, float*, double);
template bool mix_y_split<double2>(mafx_ctx*, double2*, int, bool);
template bool mix_y_split<float2>(mafx_ctx*, float2*, int, bool);

} // namespace mafx
