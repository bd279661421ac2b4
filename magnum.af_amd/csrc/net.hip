// Learned warm start for the LBFGS minimizer: a 4-level convolutional encoder-decoder (BF16
// weights, FP32 activations and accumulation), its backward pass and an Adam step, all as HIP
// kernels on the library's stream.  There is no counterpart in the reference; the CPU restatement
// that checks these kernels is oracle/warmstart_net.py (same operations, same order).
//
// Layout: activations [B][C][H][W] f32, x fastest, which for B = 1 and nz = 1 is the library's
// SoA [3][ny][nx] order of m.  Parameters: per layer W [Cout][Cin][3][3] then b [Cout], flat.
//
// Kernels:
//   k_conv            3x3 convolution as an implicit GEMM on the FP32 matrix cores, in the order of the
//                     plain loop nest; the data gradient is the same kernel on the reversed,
//                     transposed weights.  Input channel c < Ca comes from a (optionally at half
//                     resolution, read through nearest upsampling), c >= Ca from b (channel
//                     concatenation).
//   k_conv_wgrad      dW, db on FP32 MFMAs as per-chunk partials (fixed tile order per chunk), then
//                     k_reduce_chunks sums the chunks in a fixed order: deterministic.
//   pooling, upsampling and ReLU masks as small elementwise kernels; k_norm_loss normalises the
//   3-vector output per cell and forms the loss and its gradient.
#include <cmath>
#include <cstring>
#include <algorithm>
#include <random>
#include <type_traits>

#include "net.hpp"

namespace mafx {

// Where each layer's weight-gradient partials lie (k_reduce_chunks): first parameter, number of
// parameters, first partial, number of chunks.
struct GradTable {
    int64_t off[kNetLayers], count[kNetLayers], part[kNetLayers];
    int nchunk[kNetLayers];
};

struct NetAct {
    DevBuf pool;
    float *e1, *p1, *e2, *p2, *e3, *p3, *e4, *d3, *d2, *d1, *y, *m;
    float *dy, *dd1, *dupd2, *de1s, *dd2, *dupd3, *de2s, *dd3, *dupe4, *de3s, *de4, *dp3, *de3, *dp2, *de2, *dp1, *de1;
    DevBuf wpart; // weight-gradient partials of all layers
    GradTable grads;
    const float* x{nullptr};
};

namespace {

__device__ __forceinline__ uint16_t f2bf(float f) { // round to nearest even (finite inputs)
    const uint32_t u = __float_as_uint(f);
    return static_cast<uint16_t>((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// ---- convolutions on the matrix cores ------------------------------------------------------------
// A 3x3 convolution is a GEMM: M = output channels, N = pixels, K = (input channel, tap), on
// v_mfma_f32_16x16x4_f32 with the BF16 weights widened in registers.  That instruction is a chain
// of four FMAs in K order (checked bit by bit against fmaf, subnormal values included), so with K
// running over channels, then taps, every output is the sum of the plain loop nest, at twice the
// rate of its FP32 vector form: a 256 x 256 prediction takes 156 us where the vector kernels took 929,
// and a training batch of 32 films of 64 x 64 811 against 2896 us (forward convolutions 190 us, data
// gradients 167, weight gradients 223; their products alone are 94, 90 and 94 us at the matrix
// rate).  An exact split of the activations into three BF16 parts for the 16-bit matrix rate took 124 us
// for the prediction, but sums in another order: activations within rounding of zero then
// change sides of their ReLU, and gradients moved by up to 2e-4.
//
// A wave owns MT x NT tiles of 16 channels x 16 pixels; the four waves of a work-group take
// consecutive pixels and the same channels.  CC channels with their halo are staged in LDS per round,
// [channel][pixel], in two buffers: the next round's values are loaded into registers while the
// current one is multiplied, and its weights replace the current ones as they are used.
using f32x4 = __attribute__((ext_vector_type(4))) float;

// Packed weights: [group of 8 K channels][M tile][3][lane][8] BF16, zero beyond the layer's
// channels.  K entry 9 c + tap of a group is step (9 c + tap) / 4, lane group (9 c + tap) % 4;
// lane l holds row l % 16 of lane group l / 16, and its 18 steps in order (24 places).
struct PackSeg {
    int64_t woff;     // the layer's W [Cout][Cin][3][3] in the parameters
    int64_t off, end; // its packed range
    int Cin, Cout, trans;
};
struct PackTable {
    PackSeg s[2 * kNetLayers];
    int n;
};

constexpr int kPackGroup = 3 * 64 * 8; // places per group and M tile
int64_t packed_size(int Mch, int K) {
    return static_cast<int64_t>((K + 7) / 8) * ((Mch + 15) / 16) * kPackGroup;
}

// One launch rounds the masters to BF16 and lays out both forms of every layer: forward (M = Cout,
// K = Cin) and data gradient (trans: M = Cin, K = Cout, taps reversed).
__global__ void k_pack_weights(const float* __restrict__ master, uint16_t* __restrict__ packed, PackTable T) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= T.s[T.n - 1].end) return;
    int q = 0;
    while (i >= T.s[q].end) ++q;
    const PackSeg& g = T.s[q];
    const int Mch = g.trans ? g.Cin : g.Cout, K = g.trans ? g.Cout : g.Cin, mt = (Mch + 15) / 16;
    const int e = static_cast<int>(i - g.off);
    const int j = e & 7, lane = (e >> 3) & 63, r = e >> 9, step = (r % 3) * 8 + j;
    const int m = ((r / 3) % mt) * 16 + (lane & 15), kk = 4 * step + (lane >> 4);
    const int k = (r / 3 / mt) * 8 + kk / 9, tap = kk % 9;
    uint16_t v = 0;
    if (step < 18 && m < Mch && k < K) {
        const int64_t w = g.trans ? (static_cast<int64_t>(k) * g.Cin + m) * 9 + 8 - tap
                                  : (static_cast<int64_t>(m) * g.Cin + k) * 9 + tap;
        v = f2bf(master[g.woff + w]);
    }
    packed[i] = v;
}

struct ConvArgs {
    const float *a, *b; // input channels [0, Ca) from a (at half resolution when a_up), the rest from b
    int Ca, a_up, Cb;
    const uint16_t* w; // packed
    const float* bias; // or null
    const float* mask; // or null: outputs where it is not positive become 0 (layout of o1)
    float *o1, *o2;    // output channels [0, Co1) and the rest
    int Co1, Co2, H, W, tiles_x, relu, mtiles;
};

template <int MT, int NT, int CC, int TW>
__global__ void __launch_bounds__(256) k_conv(ConvArgs A) {
    constexpr int TH = 64 * NT / TW, HW_ = TW + 2, PX = HW_ * (TH + 2);
    __shared__ float stage[2][CC * PX];
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63, wave = tid >> 6;
    const int tile = static_cast<int>(blockIdx.x), mt0 = static_cast<int>(blockIdx.y) * MT;
    const int n = static_cast<int>(blockIdx.z);
    const int ty0 = (tile / A.tiles_x) * TH, tx0 = (tile % A.tiles_x) * TW;
    const int col = lane & 15, kg = lane >> 4;
    const int Ci = A.Ca + A.Cb, nchunks = (Ci + CC - 1) / CC;
    const int64_t plane = static_cast<int64_t>(A.H) * A.W, aplane = A.a_up ? plane / 4 : plane;
    const float* an = A.a + n * A.Ca * aplane;
    const float* bn = A.b + n * A.Cb * plane;

    // A lane stages PXI halo pixels of every CG-th channel.  A pixel outside the image (or a channel
    // that pads the chunk) reads a value that exists and becomes zero when it is staged, so that all
    // loads are issued without branches.
    constexpr int TPG = PX <= 128 ? 128 : 256, CG = 256 / TPG, PXI = (PX + TPG - 1) / TPG, CJ = CC / CG;
    static_assert(CC % CG == 0 && CC % 8 == 0, "whole channel groups");
    const int cg = tid / TPG, sp = tid % TPG;
    float v[PXI][CJ];
    int off[PXI], up[PXI];
    bool in[PXI];
#pragma unroll
    for (int i = 0; i < PXI; ++i) {
        const int px = sp + i * TPG, yy = ty0 + px / HW_ - 1, xx = tx0 + px % HW_ - 1;
        in[i] = px < PX && yy >= 0 && yy < A.H && xx >= 0 && xx < A.W;
        off[i] = in[i] ? yy * A.W + xx : 0;
        up[i] = in[i] && A.a_up ? (yy >> 1) * (A.W >> 1) + (xx >> 1) : off[i];
    }
    const auto fetch = [&](int c) {
        // a chunk lies in one operand: Ca is a multiple of CC where b is used
        const int cb = c * CC;
        const bool from_a = cb < A.Ca;
        const int64_t pl = from_a ? aplane : plane;
        const float* src = from_a ? an + cb * aplane : bn + (cb - A.Ca) * plane;
#pragma unroll
        for (int i = 0; i < PXI; ++i) {
            const float* q = src + (from_a ? up[i] : off[i]);
#pragma unroll
            for (int j = 0; j < CJ; ++j) v[i][j] = q[(CC > 8 || cg + CG * j < Ci ? cg + CG * j : 0) * pl];
        }
    };
    const auto put = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PXI; ++i) {
            const int px = sp + i * TPG;
            if (px >= PX) continue;
#pragma unroll
            for (int j = 0; j < CJ; ++j)
                stage[buf][(cg + CG * j) * PX + px] = in[i] && (CC > 8 || cg + CG * j < Ci) ? v[i][j] : 0.0f;
        }
    };
    uint4 w[CC / 8][MT][3];
    const uint4* wp = reinterpret_cast<const uint4*>(A.w) + mt0 * (kPackGroup / 8) + lane;
    const auto weights = [&](int c, int g) {
        const uint4* q = wp + static_cast<int64_t>(c * (CC / 8) + g) * A.mtiles * (kPackGroup / 8);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int h = 0; h < 3; ++h) w[g][m][h] = q[m * (kPackGroup / 8) + h * 64];
    };
    fetch(0);
#pragma unroll
    for (int g = 0; g < CC / 8; ++g) weights(0, g);
    float bias[MT][4];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int co = (mt0 + m) * 16 + 4 * kg + r;
            bias[m][r] = A.bias ? A.bias[co < A.Co1 + A.Co2 ? co : 0] : 0.0f;
        }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m][t] = f32x4{0, 0, 0, 0};
    // LDS offsets of this lane's K entry in each of the nine steps of a group of four channels
    int pb[9];
    {
        const int p = wave * 16 * NT + col, base = (p / TW) * HW_ + p % TW;
#pragma unroll
        for (int s = 0; s < 9; ++s) {
            const int kk = 4 * s + kg, tap = kk % 9;
            pb[s] = (kk / 9) * PX + base + (tap / 3) * HW_ + tap % 3;
        }
    }
    // The products of a staged round.  With MORE the next round's loads are in flight meanwhile; they
    // are issued without a condition (the last round is a call of its own), since a wait after a
    // join of paths with and without loads would wait for all of them.  The operands of a step are
    // read from LDS one step ahead.
    const auto products = [&](int c, auto more) {
        constexpr bool MORE = decltype(more)::value;
        if constexpr (MORE) fetch(c + 1);
        const float* sb = stage[c & 1];
        constexpr int STEPS = CC / 8 * 18;
        float x[2][NT];
        const auto read = [&](int s) {
            // N tile t starts 16 t pixels on: 16 t / TW rows
#pragma unroll
            for (int t = 0; t < NT; ++t) x[s & 1][t] = sb[pb[s % 9] + (s / 9) * 4 * PX + (16 * t / TW) * HW_];
        };
        read(0);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            if (s + 1 < STEPS) read(s + 1);
            const int g = s / 18, e = s % 18;
            float wf[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const uint4& q = w[g][m][e / 8];
                const uint32_t u = (e % 8) / 2 == 0 ? q.x : (e % 8) / 2 == 1 ? q.y : (e % 8) / 2 == 2 ? q.z : q.w;
                wf[m] = __uint_as_float(e & 1 ? u & 0xffff0000u : u << 16);
            }
            __builtin_amdgcn_sched_barrier(0); // keep the reads ahead of the products
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[m], x[s & 1][t], acc[m][t], 0, 0, 0);
            if (MORE && e == 17) weights(c + 1, g);
        }
        if constexpr (MORE) {
            put((c + 1) & 1);
            __syncthreads();
        }
    };
    put(0);
    __syncthreads();
    for (int c = 0; c + 1 < nchunks; ++c) products(c, std::true_type{});
    products(nchunks - 1, std::false_type{});
    // an M tile lies in one output: Co1 is a multiple of 16 where o2 is used
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int p = (wave * NT + t) * 16 + col, y = ty0 + p / TW, x = tx0 + p % TW;
        if (y >= A.H || x >= A.W) continue;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int ct = (mt0 + m) * 16;
            const bool first = ct < A.Co1;
            const int rows = A.Co1 + A.Co2 - ct - 4 * kg; // of this lane's four, those that exist
            const int64_t o = ((first ? static_cast<int64_t>(n) * A.Co1 + ct
                                      : static_cast<int64_t>(n) * A.Co2 + (ct - A.Co1)) + 4 * kg) * plane + y * A.W + x;
            float* dst = (first ? A.o1 : A.o2) + o;
            float mk[4] = {1.0f, 1.0f, 1.0f, 1.0f};
            if (A.mask && first)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (r < rows) mk[r] = A.mask[o + r * plane];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float f = A.bias ? acc[m][t][r] + bias[m][r] : acc[m][t][r];
                if (A.relu) f = fmaxf(f, 0.0f);
                if (!(mk[r] > 0.0f)) f = 0.0f;
                if (r < rows) dst[r * plane] = f;
            }
        }
    }
}

// Weight gradient dW[co][ci][tap] = sum over pixels d[co][p] in[ci][p + tap], as FP32 MFMAs
// (v_mfma_f32_16x16x4_f32: one K entry per lane, so a tap's shift by one pixel is only another LDS
// address, where packed 16-bit operands would need K vectors that straddle it).  Work-group: 32
// output x 32 input channels of one chunk of 128-pixel tiles; each wave 16 x 16 channels, all nine
// taps (36 accumulator registers), and every PS-th K step, PS = 2, or more where the layer has at
// most 16 channels on a side; a K step of 4 pixels reads one d and nine input operands for nine
// 32-cycle MFMAs, so LDS does not bound it.  The next tile's input is loaded into registers while
// the current one is multiplied, and the PS partial tiles are summed through LDS at the end, so that
// two waves per SIMD share one partial in memory.  db is the sum over d of the work-groups of the
// first input block.
template <int TW, int TH>
__global__ void __launch_bounds__(512)
    k_conv_wgrad(const float* __restrict__ d, int Co, const float* __restrict__ a, int Ca, int a_up,
                 const float* __restrict__ b, int Cb, int B, int H, int W, int tiles_x, int tiles_img, int nchunk,
                 float* __restrict__ part) {
    constexpr int P = TW * TH, HW_ = TW + 2, PX = HW_ * (TH + 2), SD = P + 4, SA = PX, BS = 512;
    static_assert(P == 128 && SD % 8 == 4 && SA % 8 == 4, "strides of odd multiples of 4: no bank conflicts");
    __shared__ float lds[32 * (SD + SA)];
    static_assert(sizeof(lds) >= 4 * 36 * 64 * sizeof(float), "the partial tiles of four waves");
    float *s_d = lds, *s_in = lds + 32 * SD;
    const int Ci = Ca + Cb;
    const int co0 = static_cast<int>(blockIdx.x) * 32, ci0 = static_cast<int>(blockIdx.y) * 32;
    const int chunk = static_cast<int>(blockIdx.z);
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nco = Co - co0 > 16 ? 2 : 1, nci = Ci - ci0 > 16 ? 2 : 1, PS = 8 / (nco * nci);
    const int wt = wave % (nco * nci), ps = wave / (nco * nci);
    const int wco = (wt / nci) * 16, wci = (wt % nci) * 16;
    constexpr int ND = 32 * P / BS, NA = (32 * PX + BS - 1) / BS;
    float rd[ND], ra[NA];
    // a block of 32 input channels lies in one operand (Ca is a multiple of 32 where b is used); an
    // element's offset from its tile's first pixel and its place in the halo are found once
    const bool from_a = ci0 < Ca, half = from_a && a_up;
    const int64_t plane = static_cast<int64_t>(H) * W, ap = half ? plane / 4 : plane;
    const int arow = half ? W >> 1 : W;
    int od[ND], oa[NA], pa_[NA];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const int e = tid + i * BS, o = e / P, p = e % P;
        od[i] = co0 + o < Co ? static_cast<int>(o * plane) + (p / TW) * W + p % TW : -1;
    }
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int e = tid + i * BS, c = e / PX, r = e - c * PX, y = r / HW_ - 1, x = r % HW_ - 1;
        const bool in = e < 32 * PX && ci0 + c < Ci;
        oa[i] = static_cast<int>(c * ap) + (half ? (y >> 1) * arow + (x >> 1) : y * arow + x);
        pa_[i] = in ? ((y + 1) << 8) | (x + 1) : -1;
    }
    const auto fetch = [&](int t) {
        const int n = t / tiles_img, tile = t - n * tiles_img;
        const int ty0 = (tile / tiles_x) * TH, tx0 = (tile % tiles_x) * TW;
        const float* dp = d + (static_cast<int64_t>(n) * Co + co0) * plane + ty0 * W + tx0;
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int p = (tid + i * BS) % P;
            rd[i] = od[i] >= 0 && ty0 + p / TW < H && tx0 + p % TW < W ? dp[od[i]] : 0.0f;
        }
        const float* ip = (from_a ? a + (static_cast<int64_t>(n) * Ca + ci0) * ap
                                  : b + (static_cast<int64_t>(n) * Cb + (ci0 - Ca)) * ap) +
                          (half ? (ty0 >> 1) * arow + (tx0 >> 1) : ty0 * arow + tx0);
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int y = ty0 + (pa_[i] >> 8) - 1, x = tx0 + (pa_[i] & 255) - 1;
            const bool in = pa_[i] >= 0 && static_cast<unsigned>(y) < static_cast<unsigned>(H) &&
                            static_cast<unsigned>(x) < static_cast<unsigned>(W);
            ra[i] = in ? ip[oa[i]] : 0.0f;
        }
    };
    f32x4 acc[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) acc[k] = f32x4{0, 0, 0, 0};
    float accb = 0.0f;
    const int total = B * tiles_img;
    fetch(chunk); // chunk < nchunk <= total
    const int kk = lane >> 4;
    const float* pd = s_d + (wco + (lane & 15)) * SD + kk;
    const float* pa = s_in + (wci + (lane & 15)) * SA + kk;
    for (int t = chunk; t < total; t += nchunk) {
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            const int e = tid + i * BS;
            s_d[(e / P) * SD + e % P] = rd[i];
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int e = tid + i * BS;
            if (e < 32 * PX) s_in[e] = ra[i];
        }
        __syncthreads();
        if (t + nchunk < total) fetch(t + nchunk);
        if (blockIdx.y == 0) { // 16 lanes per output channel
            const float* q = s_d + (tid >> 4) * SD + (tid & 15);
#pragma unroll
            for (int i = 0; i < P / 16; ++i) accb += q[16 * i];
        }
        // the operands of a step are read from LDS one step ahead (beyond the last one they are
        // the first step's again, unused)
        float dv[2], iv[2][9];
        const auto read = [&](int s, int h) {
            const int u = s < P / 4 ? s : 0, y = u / (TW / 4), x = (u % (TW / 4)) * 4;
            dv[h] = pd[4 * u];
            const float* q = pa + y * HW_ + x;
#pragma unroll
            for (int k = 0; k < 9; ++k) iv[h][k] = q[(k / 3) * HW_ + k % 3];
        };
        read(ps, 0);
        for (int s = ps; s < P / 4; s += 2 * PS) { // an even number of steps: P / 4 / PS = 16, 8 or 4
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                read(s + (h + 1) * PS, 1 - h);
                __builtin_amdgcn_sched_barrier(0); // keep the reads ahead of the products
#pragma unroll
                for (int k = 0; k < 9; ++k)
                    acc[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(dv[h], iv[h][k], acc[k], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // sum the PS partial tiles of each 16 x 16 block, in wave order
    f32x4* red = reinterpret_cast<f32x4*>(lds) + (wt * 9 * 64 + lane);
    for (int q = 1; q < PS; ++q) {
        if (ps == q)
#pragma unroll
            for (int k = 0; k < 9; ++k) red[k * 64] = acc[k];
        __syncthreads();
        if (ps == 0)
#pragma unroll
            for (int k = 0; k < 9; ++k) acc[k] += red[k * 64];
        __syncthreads();
    }
    // partials of this chunk: dW [Co][Ci][9], then db [Co]
    const int64_t nw = static_cast<int64_t>(Co) * Ci * 9;
    float* pw = part + chunk * (nw + Co);
    const int ci = ci0 + wci + (lane & 15);
    if (ps == 0 && ci < Ci) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int co = co0 + wco + 4 * kk + r;
            if (co >= Co) break;
#pragma unroll
            for (int k = 0; k < 9; ++k) pw[(static_cast<int64_t>(co) * Ci + ci) * 9 + k] = acc[k][r];
        }
    }
    if (blockIdx.y == 0) {
#pragma unroll
        for (int s = 8; s > 0; s >>= 1) accb += __shfl_xor(accb, s, 64);
        const int co = co0 + (tid >> 4);
        if ((tid & 15) == 0 && co < Co) pw[nw + co] = accb;
    }
}

// All layers' gradients from their chunk partials, in one launch: parameter j of a layer is the sum
// over its chunks in a fixed order (eight interleaved partial sums, whose loads are in flight together).
__global__ void k_reduce_chunks(const float* __restrict__ part, GradTable T, int64_t n, float* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int l = kNetLayers - 1;
    while (l > 0 && i < T.off[l]) --l;
    const int64_t count = T.count[l];
    const float* p = part + T.part[l] + (i - T.off[l]);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int c = 0;
    for (; c + 8 <= T.nchunk[l]; c += 8)
#pragma unroll
        for (int j = 0; j < 8; ++j) s[j] += p[(c + j) * count];
    for (; c < T.nchunk[l]; ++c) s[0] += p[c * count];
    out[i] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

// 2x2 average: out [BC][h][w] from in [BC][2h][2w]
__global__ void k_pool(const float* __restrict__ in, float* __restrict__ out, int64_t BC, int h, int w) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= BC * h * w) return;
    const int64_t bc = i / (static_cast<int64_t>(h) * w);
    const int r = static_cast<int>(i - bc * h * w), y = r / w, x = r - y * w;
    const float* p = in + (bc * 2 * h + 2 * y) * (2 * w) + 2 * x;
    out[i] = 0.25f * (p[0] + p[1] + p[2 * w] + p[2 * w + 1]);
}

// out [BC][H][W] = (pool_bwd(dpool) + skip) * (act > 0)
__global__ void k_pool_bwd_add_mask(const float* __restrict__ dpool, const float* __restrict__ skip,
                                    const float* __restrict__ act, float* __restrict__ out, int64_t BC, int H,
                                    int W) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= BC * H * W) return;
    const int64_t bc = i / (static_cast<int64_t>(H) * W);
    const int r = static_cast<int>(i - bc * H * W), y = r / W, x = r - y * W;
    float v = 0.25f * dpool[(bc * (H / 2) + y / 2) * (W / 2) + x / 2];
    if (skip) v += skip[i];
    out[i] = act[i] > 0.0f ? v : 0.0f;
}

// out [BC][h][w] = up_bwd(dfull) * (act > 0), dfull [BC][2h][2w]
__global__ void k_up_bwd_mask(const float* __restrict__ dfull, const float* __restrict__ act, float* __restrict__ out,
                              int64_t BC, int h, int w) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= BC * h * w) return;
    const int64_t bc = i / (static_cast<int64_t>(h) * w);
    const int r = static_cast<int>(i - bc * h * w), y = r / w, x = r - y * w;
    const float* p = dfull + (bc * 2 * h + 2 * y) * (2 * w) + 2 * x;
    const float v = (p[0] + p[1]) + (p[2 * w] + p[2 * w + 1]);
    out[i] = act[i] > 0.0f ? v : 0.0f;
}

constexpr float kNormEps = 1e-12f;

// m = y / sqrt(|y|^2 + eps) per cell; with a target also loss partials (per work-group) and
// dy = (dm - m (m . dm)) / n with dm = 2 (m - target) scale.
__global__ void __launch_bounds__(256)
    k_norm_loss(const float* __restrict__ y, const float* __restrict__ target, float* __restrict__ m,
                float* __restrict__ dy, int B, int HW, float scale, float* __restrict__ part) {
    __shared__ float red[256];
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    float l = 0.0f;
    if (i < static_cast<int64_t>(B) * HW) {
        const int64_t n = i / HW, p = i - n * HW;
        const int64_t o0 = (n * 3) * HW + p, o1 = o0 + HW, o2 = o1 + HW;
        const float y0 = y[o0], y1 = y[o1], y2 = y[o2];
        const float nrm = sqrtf(y0 * y0 + y1 * y1 + y2 * y2 + kNormEps);
        const float m0 = y0 / nrm, m1 = y1 / nrm, m2 = y2 / nrm;
        m[o0] = m0;
        m[o1] = m1;
        m[o2] = m2;
        if (target) {
            const float r0 = m0 - target[o0], r1 = m1 - target[o1], r2 = m2 - target[o2];
            l = r0 * r0 + r1 * r1 + r2 * r2;
            const float g0 = 2.0f * r0 * scale, g1 = 2.0f * r1 * scale, g2 = 2.0f * r2 * scale;
            const float mg = m0 * g0 + m1 * g1 + m2 * g2;
            dy[o0] = (g0 - m0 * mg) / nrm;
            dy[o1] = (g1 - m1 * mg) / nrm;
            dy[o2] = (g2 - m2 * mg) / nrm;
        }
    }
    if (!target) return;
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (static_cast<int>(threadIdx.x) < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// One work-group: 256 interleaved FP64 sums, then a fixed tree.
__global__ void __launch_bounds__(256) k_sum_f64(const float* __restrict__ part, int n, double* __restrict__ out) {
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (static_cast<int>(threadIdx.x) < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// Adam (Kingma & Ba 2015) with bias correction; bc1 = 1 - beta1^t, bc2 = 1 - beta2^t
__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ mo,
                       float* __restrict__ ve, int64_t n, float lr, float b1, float b2, float eps, float bc1, float bc2) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float m = b1 * mo[i] + (1.0f - b1) * gi;
    const float v = b2 * ve[i] + (1.0f - b2) * gi * gi;
    mo[i] = m;
    ve[i] = v;
    w[i] -= lr * (m / bc1) / (sqrtf(v / bc2) + eps);
}

__global__ void k_pack_input(const double* __restrict__ m0, int64_t N, float p0, float p1, float p2, float p3,
                             float p4, float* __restrict__ x) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= N) return;
    x[i] = static_cast<float>(m0[i]);
    x[N + i] = static_cast<float>(m0[N + i]);
    x[2 * N + i] = static_cast<float>(m0[2 * N + i]);
    x[3 * N + i] = p0;
    x[4 * N + i] = p1;
    x[5 * N + i] = p2;
    x[6 * N + i] = p3;
    x[7 * N + i] = p4;
}

// FP64 unit vectors from the network output (renormalised in FP64)
__global__ void k_unpack_output(const float* __restrict__ m, int64_t N, double* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const double a = m[i], b = m[N + i], c = m[2 * N + i];
    const double n = sqrt(a * a + b * b + c * c);
    out[i] = a / n;
    out[N + i] = b / n;
    out[2 * N + i] = c / n;
}

unsigned nblk(int64_t n, int b = 256) { return static_cast<unsigned>((n + b - 1) / b); }

} // namespace

Net::Net(hipStream_t s) : stream(s) {
    int64_t off = 0;
    for (int l = 0; l < kNetLayers; ++l) {
        woff[l] = off;
        off += static_cast<int64_t>(kNetCout[l]) * kNetCin[l] * 9;
        boff[l] = off;
        off += kNetCout[l];
    }
    nparams = off;
    master.alloc(sizeof(float) * nparams);
    int64_t poff = 0;
    for (int t = 0; t < 2; ++t)
        for (int l = 0; l < kNetLayers; ++l) {
            packoff[t][l] = poff;
            poff += t ? packed_size(kNetCin[l], kNetCout[l]) : packed_size(kNetCout[l], kNetCin[l]);
        }
    npacked = poff;
    packed.alloc(sizeof(uint16_t) * npacked);
    grad.alloc(sizeof(float) * nparams);
    adam_m.alloc(sizeof(float) * nparams);
    adam_v.alloc(sizeof(float) * nparams);
    MAFX_HIP(hipMemsetAsync(adam_m.p, 0, adam_m.bytes, stream));
    MAFX_HIP(hipMemsetAsync(adam_v.p, 0, adam_v.bytes, stream));
    scal.alloc(sizeof(double) * 4);
    MAFX_HIP(hipHostMalloc(reinterpret_cast<void**>(&host_scal), sizeof(double) * 4, hipHostMallocDefault));
    // He-normal initial weights, zero biases
    std::vector<float> h(nparams, 0.0f);
    std::mt19937_64 rng(12345);
    for (int l = 0; l < kNetLayers; ++l) {
        std::normal_distribution<double> nd(0.0, std::sqrt(2.0 / (9.0 * kNetCin[l])));
        for (int64_t i = woff[l]; i < boff[l]; ++i) h[i] = static_cast<float>(nd(rng));
    }
    set_params(h.data());
}

Net::~Net() {
    delete act;
    if (host_scal) (void)hipHostFree(host_scal);
}

void Net::set_params(const float* host) {
    MAFX_HIP(hipMemcpyAsync(master.p, host, sizeof(float) * nparams, hipMemcpyHostToDevice, stream));
    sync_bf16();
    MAFX_HIP(hipStreamSynchronize(stream));
}

void Net::get_params(float* host) const {
    MAFX_HIP(hipMemcpyAsync(host, master.p, sizeof(float) * nparams, hipMemcpyDeviceToHost, stream));
    MAFX_HIP(hipStreamSynchronize(stream));
}

void Net::sync_bf16() {
    PackTable T{};
    for (int t = 0; t < 2; ++t)
        for (int l = 0; l < kNetLayers; ++l) {
            PackSeg& g = T.s[T.n++];
            g = PackSeg{woff[l], packoff[t][l], 0, kNetCin[l], kNetCout[l], t};
            g.end = g.off + (t ? packed_size(kNetCin[l], kNetCout[l]) : packed_size(kNetCout[l], kNetCin[l]));
        }
    hipLaunchKernelGGL(k_pack_weights, dim3(nblk(npacked)), dim3(256), 0, stream, master.as<float>(),
                       packed.as<uint16_t>(), T);
    MAFX_HIP(hipGetLastError());
}

void Net::ensure_shape(int b, int h, int w) {
    require(b >= 1 && h >= 8 && w >= 8 && h % 8 == 0 && w % 8 == 0, "network input: H and W must be multiples of 8");
    require(static_cast<int64_t>(b) * 256 * h * w < (int64_t{1} << 31), "network input too large");
    if (act && b == B && h == H && w == W) return;
    delete act;
    act = new NetAct();
    B = b;
    H = h;
    W = w;
    const int64_t f = static_cast<int64_t>(b) * h * w; // cells at full resolution
    // float counts of each buffer at its resolution
    struct Item {
        float** p;
        int64_t n;
    };
    NetAct& A = *act;
    const Item items[] = {
        {&A.e1, 32 * f},      {&A.p1, 32 * f / 4},   {&A.e2, 64 * f / 4},  {&A.p2, 64 * f / 16},
        {&A.e3, 128 * f / 16}, {&A.p3, 128 * f / 64}, {&A.e4, 128 * f / 64}, {&A.d3, 64 * f / 16},
        {&A.d2, 32 * f / 4},  {&A.d1, 32 * f},       {&A.y, 3 * f},        {&A.m, 3 * f},
        {&A.dy, 3 * f},       {&A.dd1, 32 * f},      {&A.dupd2, 32 * f},   {&A.de1s, 32 * f},
        {&A.dd2, 32 * f / 4}, {&A.dupd3, 64 * f / 4}, {&A.de2s, 64 * f / 4}, {&A.dd3, 64 * f / 16},
        {&A.dupe4, 128 * f / 16}, {&A.de3s, 128 * f / 16}, {&A.de4, 128 * f / 64}, {&A.dp3, 128 * f / 64},
        {&A.de3, 128 * f / 16}, {&A.dp2, 64 * f / 16}, {&A.de2, 64 * f / 4}, {&A.dp1, 32 * f / 4},
        {&A.de1, 32 * f},
    };
    int64_t total = 0;
    for (const Item& it : items) total += (it.n + 63) / 64 * 64;
    A.pool.alloc(sizeof(float) * total);
    float* base = A.pool.as<float>();
    int64_t off = 0;
    for (const Item& it : items) {
        *it.p = base + off;
        off += (it.n + 63) / 64 * 64;
    }
    // weight-gradient partials of every layer, summed by one launch at the end of the backward pass
    GradTable& G = A.grads;
    int64_t poff = 0;
    for (int l = 0; l < kNetLayers; ++l) {
        const WgradShape g = wgrad_shape(l, b, h, w);
        G.off[l] = woff[l];
        G.count[l] = static_cast<int64_t>(kNetCout[l]) * (kNetCin[l] * 9 + 1);
        G.part[l] = poff;
        G.nchunk[l] = g.nchunk;
        poff += G.count[l] * g.nchunk;
    }
    A.wpart.alloc(sizeof(float) * poff);
    loss_part.alloc(sizeof(float) * nblk(f));
}

namespace {

struct ConvIn {
    const float* a;
    int Ca;
    int a_up;
    const float* b;
    int Cb;
};

// The largest wave tile (8, 4, 2, 1 MFMA tiles) that still gives about one wave per SIMD, so that
// the coarse levels fill the chip; smaller tiles stage more channels per round (CC), which keeps
// a round's products longer than the loads of the next.  TW = 8 for rows of at most 8 pixels.
void conv_launch(Net* net, ConvArgs A, int K) {
    A.mtiles = (A.Co1 + A.Co2 + 15) / 16;
    const int tw = A.W <= 8 ? 8 : 16;
    A.tiles_x = (A.W + tw - 1) / tw;
    const auto tiles = [&](int nt) { return A.tiles_x * ((A.H + 64 * nt / tw - 1) / (64 * nt / tw)); };
    const auto waves = [&](int mt, int nt) { return int64_t{4} * tiles(nt) * (A.mtiles / mt) * net->B; };
    constexpr int64_t kFill = 1024;
    int mt = A.mtiles % 2 == 0 ? 2 : 1, nt = 4;
    while (nt > 1 && waves(mt, nt) < kFill) nt /= 2;
    if (waves(mt, nt) < kFill) mt = 1;
    using KC = void (*)(ConvArgs);
    const auto pick = [&](auto twc) -> KC {
        constexpr int TW = decltype(twc)::value;
        const bool one = K <= 8;
        if (mt == 2) {
            if (nt == 4) return k_conv<2, 4, 8, TW>;
            if (nt == 2) return one ? k_conv<2, 2, 8, TW> : k_conv<2, 2, 16, TW>;
            return one ? k_conv<2, 1, 8, TW> : k_conv<2, 1, 32, TW>;
        }
        if (nt == 4) return k_conv<1, 4, 8, TW>;
        if (nt == 2) return one ? k_conv<1, 2, 8, TW> : k_conv<1, 2, 16, TW>;
        return one ? k_conv<1, 1, 8, TW> : k_conv<1, 1, 32, TW>;
    };
    const KC k = tw == 8 ? pick(std::integral_constant<int, 8>{}) : pick(std::integral_constant<int, 16>{});
    hipLaunchKernelGGL(k, dim3(tiles(nt), A.mtiles / mt, net->B), dim3(256), 0, net->stream, A);
    MAFX_HIP(hipGetLastError());
}

void conv_fwd(Net* net, int layer, ConvIn in, float* out, int h, int w, bool relu) {
    require(in.Ca + in.Cb == kNetCin[layer], "conv: channel mismatch");
    ConvArgs A{};
    A.a = in.a;
    A.Ca = in.Ca;
    A.a_up = in.a_up;
    A.b = in.b;
    A.Cb = in.Cb;
    A.w = net->packed.as<uint16_t>() + net->packoff[0][layer];
    A.bias = net->master.as<float>() + net->boff[layer];
    A.o1 = out;
    A.Co1 = kNetCout[layer];
    A.H = h;
    A.W = w;
    A.relu = relu ? 1 : 0;
    conv_launch(net, A, kNetCin[layer]);
}

// data gradient of layer `layer` from d (its output gradient): channels [0, C1) to o1 (zeroed where
// mask, if any, is not positive), the rest to o2
void conv_bwd_data(Net* net, int layer, const float* d, float* o1, int C1, float* o2, const float* mask, int h, int w) {
    ConvArgs A{};
    A.a = d;
    A.Ca = kNetCout[layer];
    A.w = net->packed.as<uint16_t>() + net->packoff[1][layer];
    A.mask = mask;
    A.o1 = o1;
    A.Co1 = C1;
    A.o2 = o2;
    A.Co2 = kNetCin[layer] - C1;
    A.H = h;
    A.W = w;
    conv_launch(net, A, kNetCout[layer]);
}

void conv_bwd_weight(Net* net, int layer, const float* d, ConvIn in, int h, int w) {
    NetAct& A = *net->act;
    const WgradShape g = wgrad_shape(layer, net->B, net->H, net->W);
    require(g.h == h && g.w == w, "weight gradient: level mismatch");
    const int Cin = kNetCin[layer], Cout = kNetCout[layer];
    const auto k = g.tw == 8 ? k_conv_wgrad<8, 16> : k_conv_wgrad<16, 8>;
    hipLaunchKernelGGL(k, dim3((Cout + 31) / 32, (Cin + 31) / 32, g.nchunk), dim3(512), 0, net->stream, d, Cout, in.a,
                       in.Ca, in.a_up, in.b, in.Cb, net->B, h, w, g.tiles_x, g.tiles, g.nchunk,
                       A.wpart.as<float>() + A.grads.part[layer]);
    MAFX_HIP(hipGetLastError());
}

void pool_fwd(Net* net, const float* in, float* out, int C, int h, int w) { // h, w: output size
    const int64_t n = static_cast<int64_t>(net->B) * C * h * w;
    hipLaunchKernelGGL(k_pool, dim3(nblk(n)), dim3(256), 0, net->stream, in, out, static_cast<int64_t>(net->B) * C, h, w);
}

} // namespace

void Net::forward(const float* x) {
    NetAct& A = *act;
    A.x = x;
    const int h1 = H, w1 = W, h2 = H / 2, w2 = W / 2, h3 = H / 4, w3 = W / 4, h4 = H / 8, w4 = W / 8;
    conv_fwd(this, 0, {x, 8, 0, nullptr, 0}, A.e1, h1, w1, true);
    pool_fwd(this, A.e1, A.p1, 32, h2, w2);
    conv_fwd(this, 1, {A.p1, 32, 0, nullptr, 0}, A.e2, h2, w2, true);
    pool_fwd(this, A.e2, A.p2, 64, h3, w3);
    conv_fwd(this, 2, {A.p2, 64, 0, nullptr, 0}, A.e3, h3, w3, true);
    pool_fwd(this, A.e3, A.p3, 128, h4, w4);
    conv_fwd(this, 3, {A.p3, 128, 0, nullptr, 0}, A.e4, h4, w4, true);
    conv_fwd(this, 4, {A.e4, 128, 1, A.e3, 128}, A.d3, h3, w3, true);
    conv_fwd(this, 5, {A.d3, 64, 1, A.e2, 64}, A.d2, h2, w2, true);
    conv_fwd(this, 6, {A.d2, 32, 1, A.e1, 32}, A.d1, h1, w1, true);
    conv_fwd(this, 7, {A.d1, 32, 0, nullptr, 0}, A.y, h1, w1, false);
    hipLaunchKernelGGL(k_norm_loss, dim3(nblk(static_cast<int64_t>(B) * H * W)), dim3(256), 0, stream, A.y,
                       static_cast<const float*>(nullptr), A.m, static_cast<float*>(nullptr), B, H * W, 0.0f,
                       static_cast<float*>(nullptr));
    MAFX_HIP(hipGetLastError());
}

const float* Net::output() const { return act->m; }

double Net::backward(const float* target) {
    NetAct& A = *act;
    const int h1 = H, w1 = W, h2 = H / 2, w2 = W / 2, h3 = H / 4, w3 = W / 4, h4 = H / 8, w4 = W / 8;
    const int64_t f = static_cast<int64_t>(B) * H * W;
    const unsigned nb = nblk(f);
    hipLaunchKernelGGL(k_norm_loss, dim3(nb), dim3(256), 0, stream, A.y, target, A.m, A.dy, B, H * W,
                       static_cast<float>(1.0 / static_cast<double>(f)), loss_part.as<float>());
    hipLaunchKernelGGL(k_sum_f64, dim3(1), dim3(256), 0, stream, loss_part.as<float>(), static_cast<int>(nb),
                       scal.as<double>());
    const int64_t Bl = B;
    // layer 8: y = conv(d1)
    conv_bwd_data(this, 7, A.dy, A.dd1, 32, nullptr, A.d1, h1, w1);
    conv_bwd_weight(this, 7, A.dy, {A.d1, 32, 0, nullptr, 0}, h1, w1);
    // layer 7: d1 = relu(conv(cat(up(d2), e1)))
    conv_bwd_data(this, 6, A.dd1, A.dupd2, 32, A.de1s, nullptr, h1, w1);
    conv_bwd_weight(this, 6, A.dd1, {A.d2, 32, 1, A.e1, 32}, h1, w1);
    hipLaunchKernelGGL(k_up_bwd_mask, dim3(nblk(32 * f / 4)), dim3(256), 0, stream, A.dupd2, A.d2, A.dd2, Bl * 32, h2,
                       w2);
    // layer 6: d2 = relu(conv(cat(up(d3), e2)))
    conv_bwd_data(this, 5, A.dd2, A.dupd3, 64, A.de2s, nullptr, h2, w2);
    conv_bwd_weight(this, 5, A.dd2, {A.d3, 64, 1, A.e2, 64}, h2, w2);
    hipLaunchKernelGGL(k_up_bwd_mask, dim3(nblk(64 * f / 16)), dim3(256), 0, stream, A.dupd3, A.d3, A.dd3, Bl * 64,
                       h3, w3);
    // layer 5: d3 = relu(conv(cat(up(e4), e3)))
    conv_bwd_data(this, 4, A.dd3, A.dupe4, 128, A.de3s, nullptr, h3, w3);
    conv_bwd_weight(this, 4, A.dd3, {A.e4, 128, 1, A.e3, 128}, h3, w3);
    hipLaunchKernelGGL(k_up_bwd_mask, dim3(nblk(128 * f / 64)), dim3(256), 0, stream, A.dupe4, A.e4, A.de4, Bl * 128,
                       h4, w4);
    // layer 4: e4 = relu(conv(p3))
    conv_bwd_data(this, 3, A.de4, A.dp3, 128, nullptr, nullptr, h4, w4);
    conv_bwd_weight(this, 3, A.de4, {A.p3, 128, 0, nullptr, 0}, h4, w4);
    hipLaunchKernelGGL(k_pool_bwd_add_mask, dim3(nblk(128 * f / 16)), dim3(256), 0, stream, A.dp3, A.de3s, A.e3,
                       A.de3, Bl * 128, h3, w3);
    // layer 3: e3 = relu(conv(p2))
    conv_bwd_data(this, 2, A.de3, A.dp2, 64, nullptr, nullptr, h3, w3);
    conv_bwd_weight(this, 2, A.de3, {A.p2, 64, 0, nullptr, 0}, h3, w3);
    hipLaunchKernelGGL(k_pool_bwd_add_mask, dim3(nblk(64 * f / 4)), dim3(256), 0, stream, A.dp2, A.de2s, A.e2, A.de2,
                       Bl * 64, h2, w2);
    // layer 2: e2 = relu(conv(p1))
    conv_bwd_data(this, 1, A.de2, A.dp1, 32, nullptr, nullptr, h2, w2);
    conv_bwd_weight(this, 1, A.de2, {A.p1, 32, 0, nullptr, 0}, h2, w2);
    hipLaunchKernelGGL(k_pool_bwd_add_mask, dim3(nblk(32 * f)), dim3(256), 0, stream, A.dp1, A.de1s, A.e1, A.de1,
                       Bl * 32, h1, w1);
    // layer 1: e1 = relu(conv(x))
    conv_bwd_weight(this, 0, A.de1, {A.x, 8, 0, nullptr, 0}, h1, w1);
    hipLaunchKernelGGL(k_reduce_chunks, dim3(nblk(nparams)), dim3(256), 0, stream, A.wpart.as<float>(), A.grads, nparams,
                       grad.as<float>());
    MAFX_HIP(hipGetLastError());
    MAFX_HIP(hipMemcpyAsync(host_scal, scal.p, sizeof(double), hipMemcpyDeviceToHost, stream));
    MAFX_HIP(hipStreamSynchronize(stream));
    // the partials hold sum |m - target|^2; the loss is its mean over the B H W cells
    return host_scal[0] / static_cast<double>(f);
}

void Net::adam(float lr, float beta1, float beta2, float eps) {
    ++adam_t;
    const float bc1 = static_cast<float>(1.0 - std::pow(static_cast<double>(beta1), static_cast<double>(adam_t)));
    const float bc2 = static_cast<float>(1.0 - std::pow(static_cast<double>(beta2), static_cast<double>(adam_t)));
    hipLaunchKernelGGL(k_adam, dim3(nblk(nparams)), dim3(256), 0, stream, master.as<float>(), grad.as<float>(),
                       adam_m.as<float>(), adam_v.as<float>(), nparams, lr, beta1, beta2, eps, bc1, bc2);
    MAFX_HIP(hipGetLastError());
    sync_bf16();
}

void net_pack_input(Net* net, const double* m0, int nx, int ny, const float planes[5], float* x) {
    const int64_t N = static_cast<int64_t>(nx) * ny;
    hipLaunchKernelGGL(k_pack_input, dim3(nblk(N)), dim3(256), 0, net->stream, m0, N, planes[0], planes[1], planes[2],
                       planes[3], planes[4], x);
    MAFX_HIP(hipGetLastError());
}

void net_unpack_output(Net* net, const float* m, int nx, int ny, double* m_out) {
    const int64_t N = static_cast<int64_t>(nx) * ny;
    hipLaunchKernelGGL(k_unpack_output, dim3(nblk(N)), dim3(256), 0, net->stream, m, N, m_out);
    MAFX_HIP(hipGetLastError());
}

} // namespace mafx
