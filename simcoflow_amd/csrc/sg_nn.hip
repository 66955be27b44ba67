// Convolutional encoder-decoder of the learned warm start: forward,
// backward (data and weight gradients) and Adam, hand-written for the
// gfx950 matrix cores.  Convolutions are implicit GEMMs on
// v_mfma_f32_16x16x32_bf16: the output tile is 16 channels x 16 pixels, the
// reduction runs over (tap, input channel) in chunks of 32, activations are
// channel-innermost so one lane's 8 consecutive reduction elements are one
// 16-byte load.  Weight gradients reduce over pixels: the same loads are
// transposed in registers, 8 lanes at a time, so a lane holds 8 consecutive
// pixels of a channel.  No counterpart in the reference (it starts PCG from
// zero, ProjectionP_Mod.f90:319).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "sg_nn.hpp"

namespace sg {
namespace nn {

namespace {

typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

enum Epi { E_RELU = 0, E_RELU_SKIP, E_OUT, E_MASK, E_PLAIN };

__device__ __forceinline__ floatx4 mfma(const bf16x8& a, const bf16x8& b, const floatx4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The results of MB x NPB tiles of channels c0.. and pixels x0.. of one row: a
// lane holds D[co = mb*16 + 4*q4 + r][px = x0 + q*16 + r16], r = 0..3.  Applies
// ReLU (optionally after adding a skip tensor), masks by aux > 0 (data gradient
// through a ReLU), writes plain, or writes channel 0 as FP32 (the output layer).
template <int MB, int NPB>
__device__ __forceinline__ void conv_store(const floatx4 (&acc)[MB][NPB], const T4& in, const T4& out, const T4& aux,
                                           float* __restrict__ yo, int epi, int c0, int b, int y, int x0) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4;
#pragma unroll
    for (int q = 0; q < NPB; ++q) {
        const int px = x0 + q * 16 + r16;
        if (epi == E_OUT) {
            if (q4 == 0) yo[((size_t)b * in.H + y) * in.W + px] = acc[0][q][0];
            continue;
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int co = c0 + mb * 16 + 4 * q4;
            float v[4] = {acc[mb][q][0], acc[mb][q][1], acc[mb][q][2], acc[mb][q][3]};
            if (epi == E_RELU_SKIP || epi == E_MASK) {
                const bf16x4 a = *(const bf16x4*)(aux.p + t4off(aux, b, y + 1, px + 1) + co);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float av = (float)a[r];
                    v[r] = epi == E_MASK ? (av > 0.f ? v[r] : 0.f) : v[r] + av;
                }
            }
            if (epi == E_RELU || epi == E_RELU_SKIP) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = v[r] > 0.f ? v[r] : 0.f;
            }
            bf16x4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = (bf16)v[r];
            *(bf16x4*)(out.p + t4off(out, b, y + 1, px + 1) + co) = o;
        }
    }
}

// out(b,y,x,co) = sum_{tap,ci} wt[co][tap*CIN+ci] * in(b, y+dy-1, x+dx-1, ci)
// One wave: 16*NPB pixels of one row and COUT/CG of the output channels
// (CG > 1 on small levels, where one wave per pixel group would leave most
// of the chip idle; each output still sums over (tap, ci) in the same
// order).
template <int CIN, int COUT, int NPB, int CG>
__global__ void __launch_bounds__(256) k_conv(T4 in, const bf16* __restrict__ wt, T4 out, T4 aux,
                                              float* __restrict__ yo, int nb, int epi) {
    constexpr int KP = kpad(CIN);
    constexpr int MB = COUT / 16 / CG;
    static_assert(COUT % (16 * CG) == 0, "channel groups must split the 16-channel blocks");
    const int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4;
    const int tiles = in.W / (16 * NPB);
    const long wave_all = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wave_all >= (long)nb * in.H * tiles * CG) return;
    const int g = (int)(wave_all % CG);
    const long wave = wave_all / CG;
    if (epi == E_OUT && g != 0) return;  // the output layer keeps channel 0 only
    const int tx = (int)(wave % tiles);
    const long t = wave / tiles;
    const int y = (int)(t % in.H), b = (int)(t / in.H);
    const int x0 = tx * 16 * NPB;
    floatx4 acc[MB][NPB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int q = 0; q < NPB; ++q) acc[mb][q] = floatx4{0.f, 0.f, 0.f, 0.f};
    const bf16* wrow = wt + ((size_t)g * MB * 16 + r16) * KP + 8 * q4;
    for (int kc = 0; kc < KP; kc += 32) {
        const int k0 = kc + 8 * q4;
        const int tap = k0 / CIN, ci = k0 - tap * CIN;
        bf16x8 bv[NPB];
        if (tap < 9) {
            const int dy = tap / 3, dx = tap - 3 * dy;
            const bf16* src = in.p + t4off(in, b, y + dy, x0 + r16 + dx) + ci;
#pragma unroll
            for (int q = 0; q < NPB; ++q) bv[q] = *(const bf16x8*)(src + (size_t)q * 16 * CIN);
        } else {
#pragma unroll
            for (int q = 0; q < NPB; ++q)
#pragma unroll
                for (int e = 0; e < 8; ++e) bv[q][e] = (bf16)0.f;
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const bf16x8 av = *(const bf16x8*)(wrow + (size_t)mb * 16 * KP + kc);
#pragma unroll
            for (int q = 0; q < NPB; ++q) acc[mb][q] = mfma(av, bv[q], acc[mb][q]);
        }
    }
    conv_store<MB, NPB>(acc, in, out, aux, yo, epi, g * MB * 16, b, y, x0);
}

// k_conv for many pixels: a wave takes a strip of 16 NPB pixels by `rows` rows,
// and 16 MB channels.  A row of the input is loaded once and multiplied into
// the three output rows it belongs to, so a strip loads rows + 2 rows where
// k_conv loads 3 rows' worth for each; the weights of the workgroup's channels
// stand in LDS in the order the MFMA takes them (one 16-byte read a lane, no
// conflicts), where k_conv reads them again from the caches for every row.
// Chunks of the reduction do not run over the end of a tap row: 3 x 8 channels
// fill 24 of 32, 3 x 16 take two chunks.
//
// At 16 images, us a layer against k_conv: 16 x 16 at 256^2 24.1 / 26.6, 32 x 16
// 30.3 / 40.4, 32 x 32 at 128^2 18.1 / 20.9, 32 x 64 25.3 / 42.0, 64 x 32 (with the
// skip) 40.5 / 57, 64 x 64 at 64^2 22.5 / 28.5, 128 x 64 39.9 / 52.2, 64 x 128 34.6 /
// 41.4, 128 x 128 at 32^2 30.1 / 42.7.  The narrow layers are bound by their
// activations' bytes (2.7 TB/s at 24.1 us), the wide ones by the loads' latency at two
// waves a SIMD.
template <int CIN>
struct StripK {
    static constexpr int FR = CIN == 8 ? 1 : CIN == 16 ? 2 : 3 * CIN / 32;  // chunks of a tap row
    // column tap (3: none) and first channel of a lane's 8 in chunk f
    __host__ __device__ static constexpr int dx(int f, int q4) {
        return CIN == 8 ? q4 : CIN == 16 ? (f == 0 ? q4 >> 1 : (q4 < 2 ? 2 : 3)) : f / (CIN >= 32 ? CIN / 32 : 1);
    }
    __host__ __device__ static constexpr int ci(int f, int q4) {
        return CIN == 8 ? 0 : CIN == 16 ? 8 * (q4 & 1) : f % (CIN >= 32 ? CIN / 32 : 1) * 32 + 8 * q4;
    }
};
template <int CIN, int COUT, int MB, int NPB>
__global__ void __launch_bounds__(256, 2) k_conv_strip(T4 in, const bf16* __restrict__ wt, T4 out, T4 aux,
                                                    float* __restrict__ yo, int nb, int epi, int rows) {
    using K = StripK<CIN>;
    constexpr int FR = K::FR, KP = kpad(CIN), CG = COUT / 16 / MB;
    constexpr bool AHEAD = FR * NPB <= 12;  // the next row's loads in flight
    static_assert(COUT % (16 * MB) == 0, "channel groups must split the 16-channel blocks");
    __shared__ bf16x8 ws[3 * FR * MB * 64];
    const int lane = threadIdx.x & 63, r16 = lane & 15, q4 = lane >> 4;
    const int g = (int)(blockIdx.x % CG);
    const bf16x8 zero = {(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f};
    for (int e = threadIdx.x; e < 3 * FR * MB * 64; e += 256) {
        const int l = e & 63, f = e >> 6, mb = f % MB, fr = f / MB % FR, dy = f / MB / FR;
        const int dx = K::dx(fr, l >> 4), ci = K::ci(fr, l >> 4);
        const int co = (g * MB + mb) * 16 + (l & 15);
        ws[e] = dx < 3 ? *(const bf16x8*)(wt + (size_t)co * KP + (dy * 3 + dx) * CIN + ci) : zero;
    }
    __syncthreads();
    const int tiles = in.W / (16 * NPB), segs = (in.H + rows - 1) / rows;
    const long strip = (long)(blockIdx.x / CG) * 4 + (threadIdx.x >> 6);
    if (strip >= (long)nb * segs * tiles) return;
    const int x0 = (int)(strip % tiles) * (16 * NPB);
    const long t = strip / tiles;
    const int y0 = (int)(t % segs) * rows, b = (int)(t / segs);
    const int n = min(rows, in.H - y0);
    const bf16* src = in.p + t4off(in, b, y0, x0 + r16);
    const long step = (long)(in.W + 2) * CIN;
    auto load = [&](int iy, bf16x8 (&v)[FR][NPB]) {
#pragma unroll
        for (int f = 0; f < FR; ++f) {
            const int dx = K::dx(f, q4);
            const bf16* p = src + iy * step + (dx < 3 ? dx * CIN : 0) + K::ci(f, q4);
#pragma unroll
            for (int q = 0; q < NPB; ++q) v[f][q] = CIN >= 32 || dx < 3 ? *(const bf16x8*)(p + q * 16 * CIN) : zero;
        }
    };
    typedef floatx4 Acc[MB][NPB];
    auto clear = [&](Acc& a) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int q = 0; q < NPB; ++q) a[mb][q] = floatx4{0.f, 0.f, 0.f, 0.f};
    };
    auto add = [&](int dy, const bf16x8 (&v)[FR][NPB], Acc& a) {
#pragma unroll
        for (int f = 0; f < FR; ++f)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const bf16x8 av = ws[((dy * FR + f) * MB + mb) * 64 + lane];
#pragma unroll
                for (int q = 0; q < NPB; ++q) a[mb][q] = mfma(av, v[f][q], a[mb][q]);
            }
    };
    Acc acc[3];
    bf16x8 cur[FR][NPB], nxt[AHEAD ? FR : 1][AHEAD ? NPB : 1];
    // input row iy of the strip: tap row 0 of output row iy, 1 of iy - 1, 2 of iy - 2
    auto row = [&](int iy, Acc& a, Acc& m, Acc& z) {
        if (iy > n + 1) return;
        if constexpr (AHEAD) {
#pragma unroll
            for (int f = 0; f < FR; ++f)
#pragma unroll
                for (int q = 0; q < NPB; ++q) cur[f][q] = nxt[f][q];
            if (iy <= n) load(iy + 1, nxt);
        } else {
            load(iy, cur);
        }
        if (iy >= 2) add(2, cur, z);
        if (iy >= 1 && iy <= n) add(1, cur, m);
        if (iy >= 2) conv_store<MB, NPB>(z, in, out, aux, yo, epi, g * MB * 16, b, y0 + iy - 2, x0);
        if (iy < n) {
            clear(a);
            add(0, cur, a);
        }
    };
    if constexpr (AHEAD) load(0, nxt);
    for (int iy = 0; iy < n + 2; iy += 3) {
        row(iy, acc[0], acc[2], acc[1]);
        row(iy + 1, acc[1], acc[0], acc[2]);
        row(iy + 2, acc[2], acc[1], acc[0]);
    }
}

// 8 lanes that each hold 8 channels of one pixel (pixel = lane % 8) to 8 lanes
// that each hold one channel (channel = lane % 8) of the 8 pixels, in three
// exchanges: between lanes 4, 2 and 1 apart.  Moves bits only.
__device__ __forceinline__ bf16x8 transpose8(const bf16x8& v) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 u = __builtin_bit_cast(u32x4, v);
    const int lane = __lane_id();
    const bool m2 = lane & 2;
    constexpr int SHL4 = 0x104, SHR4 = 0x114, XOR2 = 0x4E, XOR1 = 0xB1;  // DPP row_shl:4, row_shr:4, quad_perm
    auto dpp = [](unsigned old, unsigned src, auto ctrl, auto banks) {
        return (unsigned)__builtin_amdgcn_update_dpp((int)old, (int)src, decltype(ctrl)::value, 0xF,
                                                     decltype(banks)::value, false);
    };
    using std::integral_constant;
    // channels 0-3 stay with lanes 0-3 (banks 0, 2), 4-7 with lanes 4-7: a = pixel lane % 4, b = four pixels on
    const integral_constant<int, SHR4> shr{};
    const integral_constant<int, SHL4> shl{};
    const integral_constant<int, 0xA> upper{};
    const integral_constant<int, 0x5> lower{};
    const unsigned a0 = dpp(u[0], u[2], shr, upper), a1 = dpp(u[1], u[3], shr, upper);
    const unsigned b0 = dpp(u[2], u[0], shl, lower), b1 = dpp(u[3], u[1], shl, lower);
    // a channel pair a lane: of pixels p, p + 2, p + 4, p + 6, p = lane % 2
    auto quad = [&](unsigned src, auto ctrl) { return dpp(0u, src, ctrl, integral_constant<int, 0xF>{}); };
    const integral_constant<int, XOR2> x2{};
    const integral_constant<int, XOR1> x1{};
    const unsigned ta = quad(m2 ? a0 : a1, x2), tb = quad(m2 ? b0 : b1, x2);
    const unsigned w[4] = {m2 ? ta : a0, m2 ? a1 : ta, m2 ? tb : b0, m2 ? b1 : tb};
    // one channel a lane: even lanes the low halves, odd lanes the high ones
    const unsigned sel = (lane & 1) ? 0x03020706u : 0x05040100u;
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = __builtin_amdgcn_perm(quad(w[k], x1), w[k], sel);
    return __builtin_bit_cast(bf16x8, o);
}

// dW[co][tap*CIN+ci] += sum_px P(px, co) * X(px shifted by tap, ci)
//
// A wave takes 16 * MBW output channels and 16 input channels, and a strip of
// 32 pixels by `rows` rows: the reduction of one MFMA is the 32 pixels of a
// row.  Activations are channel-innermost and the MFMA wants pixels innermost,
// so each 16-byte load is transposed in registers; a row of X (three shifts of
// it) serves the three taps above each other, so it is loaded and transposed
// once and kept for three rows of P.  Per row that is 3 + MBW loads and
// transposes for 9 * MBW MFMAs, the next row's loads in flight meanwhile, and
// no barrier until the strip ends.  Waves of a workgroup with the same channels
// add up in LDS before their atomics.  Measured at 16 x 256 x 256 pixels, 16 x
// 16 channels: 28 us for 67 MB, 2.4 TB/s; one tap a workgroup, with 32-pixel
// tiles transposed through LDS by 2-byte writes and two barriers a tile, took
// 254 us.
//
// TR: the tap rows a wave takes, all 3, or 1 (blockIdx.y) on levels too small to
// fill the chip: a third of the chain of transposes and sums, for three times the
// loads and waves.  16 x 16 channels at 16 x 128 pixels: 3.6 us, 5.9 with all
// three tap rows, 10.1 with those and strips no shorter than 8 rows.
template <int CIN, int COUT>
struct DwSplit {
    static constexpr int MBW = COUT >= 32 ? 2 : 1;
    static constexpr int NBK = (CIN + 15) / 16;
    static constexpr int PAIRS = COUT / 16 / MBW * NBK;  // (output, input) channel groups
};
template <int CIN, int COUT, int TR>
__global__ void __launch_bounds__(256) k_dw(T4 X, T4 P, float* __restrict__ dW, int nb, int rows) {
    using S = DwSplit<CIN, COUT>;
    constexpr int MBW = S::MBW, KP = kpad(CIN), PAIRS = S::PAIRS;
    constexpr int PB = PAIRS < 4 ? PAIRS : 4;  // channel groups in a workgroup
    constexpr int SHARE = 4 / PB;              // waves of a workgroup with the same one
    constexpr int TAPS = 3 * TR, NACC = TAPS * MBW * 4;
    static_assert(PAIRS < 4 ? 4 % PAIRS == 0 : PAIRS % 4 == 0, "waves must divide among the channel groups");
    __shared__ float part[SHARE > 1 ? 4 * NACC * 64 : 1];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r16 = lane & 15, q4 = lane >> 4;
    const long wid = (long)blockIdx.x * 4 + wv;
    const int pair = (int)(wid % PAIRS);
    const long strip = wid / PAIRS;
    const int c0 = pair % S::NBK * 16, co0 = pair / S::NBK * (16 * MBW);
    const int chunks = (P.W + 31) / 32, segs = (P.H + rows - 1) / rows;
    const int dy0 = TR == 1 ? (int)blockIdx.y : 0;
    floatx4 acc[TAPS][MBW];
#pragma unroll
    for (int k = 0; k < TAPS; ++k)
#pragma unroll
        for (int m = 0; m < MBW; ++m) acc[k][m] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (strip < (long)nb * segs * chunks) {
        const int x = (int)(strip % chunks) * 32 + 8 * q4 + (r16 & 7);
        const long t = strip / chunks;
        const int y0 = (int)(t % segs) * rows, b = (int)(t / segs);
        const int y1 = min(y0 + rows, P.H);
        const int half = 8 * (r16 >> 3);
        // pixels past the row's end and channels past the last one read as zero
        const bool okp = x < P.W, okx = okp && c0 + half < CIN;
        const bf16* pp = P.p + t4off(P, b, y0 + 1, okp ? x + 1 : 0) + co0 + half;
        const bf16* px = X.p + t4off(X, b, y0 + dy0, okx ? x : 0) + c0 + (okx ? half : 0);
        const long ps = (long)(P.W + 2) * COUT, xs = (long)(X.W + 2) * CIN;
        const bf16x8 zero = {(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f};
        bf16x8 rx[3], rp[MBW], xr[3][3];
        auto load_x = [&](int row, bf16x8 (&to)[3]) {
#pragma unroll
            for (int d = 0; d < 3; ++d) to[d] = okx ? *(const bf16x8*)(px + row * xs + d * CIN) : zero;
        };
        auto load_p = [&](int row) {
#pragma unroll
            for (int m = 0; m < MBW; ++m) rp[m] = okp ? *(const bf16x8*)(pp + row * ps + 16 * m) : zero;
        };
        auto turn_x = [&](const bf16x8 (&from)[3], bf16x8 (&to)[3]) {
#pragma unroll
            for (int d = 0; d < 3; ++d) to[d] = transpose8(from[d]);
        };
        const int n = y1 - y0;
        auto turn_p = [&](bf16x8 (&to)[MBW]) {
#pragma unroll
            for (int m = 0; m < MBW; ++m) to[m] = transpose8(rp[m]);
        };
        if constexpr (TR == 3) {
            load_x(0, xr[0]);
            load_x(1, xr[1]);
            load_x(2, rx);
            load_p(0);
            turn_x(xr[0], xr[0]);
            turn_x(xr[1], xr[1]);
            // row r of the strip: X rows r, r + 1, r + 2 sit in xr[i], xr[i + 1], xr[i + 2] (mod 3)
            auto row = [&](int r, bf16x8 (&xa)[3], bf16x8 (&xb)[3], bf16x8 (&xc)[3]) {
                if (r >= n) return;
                turn_x(rx, xc);
                bf16x8 pa[MBW];
                turn_p(pa);
                if (r + 1 < n) {
                    load_x(r + 3, rx);
                    load_p(r + 1);
                }
#pragma unroll
                for (int m = 0; m < MBW; ++m)
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        acc[d][m] = mfma(pa[m], xa[d], acc[d][m]);
                        acc[3 + d][m] = mfma(pa[m], xb[d], acc[3 + d][m]);
                        acc[6 + d][m] = mfma(pa[m], xc[d], acc[6 + d][m]);
                    }
            };
            for (int r = 0; r < n; r += 3) {
                row(r, xr[0], xr[1], xr[2]);
                row(r + 1, xr[1], xr[2], xr[0]);
                row(r + 2, xr[2], xr[0], xr[1]);
            }
        } else {
            load_x(0, rx);
            load_p(0);
            for (int r = 0; r < n; ++r) {
                bf16x8 pa[MBW];
                turn_x(rx, xr[0]);
                turn_p(pa);
                if (r + 1 < n) {
                    load_x(r + 1, rx);
                    load_p(r + 1);
                }
#pragma unroll
                for (int m = 0; m < MBW; ++m)
#pragma unroll
                    for (int d = 0; d < 3; ++d) acc[d][m] = mfma(pa[m], xr[0][d], acc[d][m]);
            }
        }
    }
    auto put = [&](int k, int m, int r, int ln, int pr, float v) {
        const int ci = pr % S::NBK * 16 + (ln & 15);
        const int co = pr / S::NBK * (16 * MBW) + m * 16 + 4 * (ln >> 4) + r;
        if (ci < CIN) atomicAdd(dW + (size_t)co * KP + (3 * dy0 + k) * CIN + ci, v);
    };
    if constexpr (SHARE > 1) {
        float* mine = part + wv * NACC * 64 + lane;
#pragma unroll
        for (int k = 0; k < TAPS; ++k)
#pragma unroll
            for (int m = 0; m < MBW; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) mine[((k * MBW + m) * 4 + r) * 64] = acc[k][m][r];
        __syncthreads();
        for (int e = tid; e < PB * NACC * 64; e += 256) {
            const int ln = e & 63, q = e >> 6, i = q % NACC;
            float v = part[e];
#pragma unroll
            for (int w = 1; w < SHARE; ++w) v += part[w * PB * NACC * 64 + e];
            put(i / (4 * MBW), i / 4 % MBW, i % 4, ln, q / NACC, v);
        }
    } else {
#pragma unroll
        for (int k = 0; k < TAPS; ++k)
#pragma unroll
            for (int m = 0; m < MBW; ++m)
#pragma unroll
                for (int r = 0; r < 4; ++r) put(k, m, r, lane, pair, acc[k][m][r]);
    }
}

// 2x2 average pooling, 8 channels per thread
__global__ void __launch_bounds__(256) k_pool(T4 in, T4 out, int nb) {
    const int c8n = out.C / 8;
    const long n = (long)nb * out.H * out.W * c8n;
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int c8 = (int)(e % c8n) * 8;
    long t = e / c8n;
    const int x = (int)(t % out.W);
    t /= out.W;
    const int y = (int)(t % out.H), b = (int)(t / out.H);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int a = 0; a < 2; ++a)
        for (int c = 0; c < 2; ++c) {
            const bf16x8 v = *(const bf16x8*)(in.p + t4off(in, b, 2 * y + a + 1, 2 * x + c + 1) + c8);
#pragma unroll
            for (int k = 0; k < 8; ++k) s[k] += (float)v[k];
        }
    bf16x8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = (bf16)(0.25f * s[k]);
    *(bf16x8*)(out.p + t4off(out, b, y + 1, x + 1) + c8) = o;
}

// nearest-neighbour upsampling by 2
__global__ void __launch_bounds__(256) k_up(T4 in, T4 out, int nb) {
    const int c8n = out.C / 8;
    const long n = (long)nb * out.H * out.W * c8n;
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int c8 = (int)(e % c8n) * 8;
    long t = e / c8n;
    const int x = (int)(t % out.W);
    t /= out.W;
    const int y = (int)(t % out.H), b = (int)(t / out.H);
    *(bf16x8*)(out.p + t4off(out, b, y + 1, x + 1) + c8) =
        *(const bf16x8*)(in.p + t4off(in, b, y / 2 + 1, x / 2 + 1) + c8);
}

// gradient through nearest upsampling and the ReLU of its input:
// P(y,x) = sum_{2x2} d(2y+a, 2x+c) * (act(y,x) > 0)
__global__ void __launch_bounds__(256) k_upT_mask(T4 d, T4 act, T4 P, int nb) {
    const int c8n = P.C / 8;
    const long n = (long)nb * P.H * P.W * c8n;
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int c8 = (int)(e % c8n) * 8;
    long t = e / c8n;
    const int x = (int)(t % P.W);
    t /= P.W;
    const int y = (int)(t % P.H), b = (int)(t / P.H);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int a = 0; a < 2; ++a)
        for (int c = 0; c < 2; ++c) {
            const bf16x8 v = *(const bf16x8*)(d.p + t4off(d, b, 2 * y + a + 1, 2 * x + c + 1) + c8);
#pragma unroll
            for (int k = 0; k < 8; ++k) s[k] += (float)v[k];
        }
    const bf16x8 m = *(const bf16x8*)(act.p + t4off(act, b, y + 1, x + 1) + c8);
    bf16x8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = (bf16)((float)m[k] > 0.f ? s[k] : 0.f);
    *(bf16x8*)(P.p + t4off(P, b, y + 1, x + 1) + c8) = o;
}

// gradient at a tensor that feeds a skip and a 2x2 pooling, through its
// ReLU: P = (skip + dd(y/2,x/2)/4) * (act > 0)
__global__ void __launch_bounds__(256) k_poolT_add_mask(T4 dd, T4 skip, T4 act, T4 P, int nb) {
    const int c8n = P.C / 8;
    const long n = (long)nb * P.H * P.W * c8n;
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int c8 = (int)(e % c8n) * 8;
    long t = e / c8n;
    const int x = (int)(t % P.W);
    t /= P.W;
    const int y = (int)(t % P.H), b = (int)(t / P.H);
    const bf16x8 a = *(const bf16x8*)(dd.p + t4off(dd, b, y / 2 + 1, x / 2 + 1) + c8);
    const bf16x8 s = *(const bf16x8*)(skip.p + t4off(skip, b, y + 1, x + 1) + c8);
    const bf16x8 m = *(const bf16x8*)(act.p + t4off(act, b, y + 1, x + 1) + c8);
    bf16x8 o;
#pragma unroll
    for (int k = 0; k < 8; ++k) o[k] = (bf16)((float)m[k] > 0.f ? (float)s[k] + 0.25f * (float)a[k] : 0.f);
    *(bf16x8*)(P.p + t4off(P, b, y + 1, x + 1) + c8) = o;
}

// loss = sum mask*(y-t)^2 / n ; gout channel 0 = 2 mask (y-t) / n.  A workgroup
// takes `per` times 256 pixels: a large batch is bound by the adds to the one sum,
// one a workgroup (16 x 256 x 256 pixels, 256 each: 57.6 us; 2048: 21.9), a small
// one by the chain of a thread's pixels (16 x 128, 256 each: 3.5 us; 2048: 8.6).
__global__ void __launch_bounds__(256) k_loss(const float* __restrict__ y, const float* __restrict__ t,
                                              const float* __restrict__ m, T4 g, int nb, float inv_n, int per,
                                              float* __restrict__ loss) {
    __shared__ float red[4];
    const long n = (long)nb * g.H * g.W;
    float l = 0.f;
    for (int k = 0; k < per; ++k) {
        const long e = ((long)blockIdx.x * per + k) * 256 + threadIdx.x;
        if (e >= n) break;
        const int x = (int)(e % g.W);
        const long r = e / g.W;
        const int yy = (int)(r % g.H), b = (int)(r / g.H);
        const float d = m[e] > 0.f ? y[e] - t[e] : 0.f;
        l += d * d * inv_n;
        g.p[t4off(g, b, yy + 1, x + 1)] = (bf16)(2.f * d * inv_n);
    }
    for (int o = 32; o >= 1; o >>= 1) l += __shfl_xor(l, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss, red[0] + red[1] + red[2] + red[3]);
}

__global__ void __launch_bounds__(256) k_fill(float* __restrict__ a, size_t n, float v) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e < n) a[e] = v;
}

__global__ void __launch_bounds__(256) k_to_bf16(const float* __restrict__ a, bf16* __restrict__ o, size_t n) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e < n) o[e] = (bf16)a[e];
}

// data-gradient weights of one layer: wf[ci][tap'*cout + co] =
// wt[co][(8-tap')*cin + ci], zero beyond 9*cout
__global__ void __launch_bounds__(256) k_flip(const bf16* __restrict__ wt, bf16* __restrict__ wf, int cin,
                                              int cout) {
    const int kpo = kpad(cout), kpi = kpad(cin);
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= cin * kpo) return;
    const int ci = e / kpo, k = e - ci * kpo;
    bf16 v = (bf16)0.f;
    if (k < 9 * cout) {
        const int tp = k / cout, co = k - tp * cout;
        v = wt[(size_t)co * kpi + (8 - tp) * cin + ci];
    }
    wf[e] = v;
}

__global__ void __launch_bounds__(256) k_adam(float* __restrict__ w, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, size_t n, float lr,
                                              float b1, float b2, float c1, float c2, float eps) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const float gg = g[e];
    const float mm = b1 * m[e] + (1.f - b1) * gg;
    const float vv = b2 * v[e] + (1.f - b2) * gg * gg;
    m[e] = mm;
    v[e] = vv;
    w[e] -= lr * (mm * c1) / (sqrtf(vv * c2) + eps);
}

inline unsigned blocks(long n) { return (unsigned)((n + 255) / 256); }

template <int CIN, int COUT, int NPB, int CG>
void conv_launch(Net* n, T4 in, const bf16* w, T4 out, T4 aux, float* yo, int nb, int epi, long waves) {
    hipLaunchKernelGGL((k_conv<CIN, COUT, NPB, CG>), dim3((unsigned)((waves * CG + 3) / 4)), dim3(256), 0, n->stream,
                       in, w, out, aux, yo, nb, epi);
}

template <int CIN, int COUT, int NPB>
void conv_split(Net* n, T4 in, const bf16* w, T4 out, T4 aux, float* yo, int nb, int epi, long waves) {
    // split the output channels while there are fewer than ~4 waves per CU
    constexpr int MB = COUT / 16;
    int cg = 1;
    while (cg < MB && waves * cg < 1024) cg *= 2;
    if (cg >= 8 && MB % 8 == 0)
        conv_launch<CIN, COUT, NPB, (MB % 8 == 0 ? 8 : 1)>(n, in, w, out, aux, yo, nb, epi, waves);
    else if (cg >= 4 && MB % 4 == 0)
        conv_launch<CIN, COUT, NPB, (MB % 4 == 0 ? 4 : 1)>(n, in, w, out, aux, yo, nb, epi, waves);
    else if (cg >= 2 && MB % 2 == 0)
        conv_launch<CIN, COUT, NPB, (MB % 2 == 0 ? 2 : 1)>(n, in, w, out, aux, yo, nb, epi, waves);
    else
        conv_launch<CIN, COUT, NPB, 1>(n, in, w, out, aux, yo, nb, epi, waves);
}

// Strips of as many rows as leave STRIP_WAVES waves, two a SIMD: with 4096 and
// 8192 a 16 x 16 layer of 16 x 256 x 256 pixels takes 26.5 and 28.1 us against
// 24.4, a 32 x 32 one of 16 x 128 x 128 22.7 and 22.7 against 18.3.  64-pixel
// strips where those can be two rows high; else, for the layers whose work per
// pixel is large, 32-pixel ones (64 x 64 at 16 x 64 x 64: 22.5 against 28.5 us),
// one row high if need be (128 x 128 at 16 x 32 x 32: 30.1 against k_conv's 42.7)
// where the channels come to 64 or more (64 x 32 at 16 x 64 x 64: 17.3 against
// 16.5).  With fewer tiles k_conv, which splits the channels further, keeps the chip
// fuller.  Layers of fewer channels are on the two finest levels only, whose widths
// are multiples of 64.
constexpr long STRIP_WAVES = 2048;

template <int CIN, int COUT, int MB, int NPB>
bool conv_strip(Net* n, T4 in, const bf16* w, T4 out, T4 aux, float* yo, int nb, int epi, long least) {
    constexpr int CG = COUT / 16 / MB;
    const long tiles = in.W / (16 * NPB), all = nb * in.H * tiles * CG;
    if (in.W % (16 * NPB) || all < least) return false;
    const int rows = (int)std::min(16l, all / STRIP_WAVES);
    const long strips = nb * ((in.H + rows - 1) / rows) * tiles;
    hipLaunchKernelGGL((k_conv_strip<CIN, COUT, MB, NPB>), dim3((unsigned)((strips + 3) / 4 * CG)), dim3(256), 0,
                       n->stream, in, w, out, aux, yo, nb, epi, rows);
    return true;
}

template <int CIN, int COUT>
int conv(Net* n, T4 in, const bf16* w, T4 out, T4 aux, float* yo, int nb, int epi) {
    constexpr int MB = COUT == 16 ? 1 : 2;
    bool strip = false;
    if constexpr (CIN < 128) strip = conv_strip<CIN, COUT, MB, 4>(n, in, w, out, aux, yo, nb, epi, 2 * STRIP_WAVES);
    if constexpr (CIN >= 64 || COUT >= 64)
        if (!strip && (CIN >= 64 || in.W % 64))
            strip = conv_strip<CIN, COUT, MB, 2>(n, in, w, out, aux, yo, nb, epi, (COUT >= 64 ? 1 : 2) * STRIP_WAVES);
    if (strip) {
        SG_HIP(hipGetLastError());
        return SG_OK;
    }
    // four 16-pixel groups per wave where that still leaves ~4 waves per CU
    if (in.W % 64 == 0 && (long)nb * in.H * (in.W / 64) >= 1024)
        conv_split<CIN, COUT, 4>(n, in, w, out, aux, yo, nb, epi, (long)nb * in.H * (in.W / 64));
    else
        conv_split<CIN, COUT, 1>(n, in, w, out, aux, yo, nb, epi, (long)nb * in.H * (in.W / 16));
    SG_HIP(hipGetLastError());
    return SG_OK;
}

// Strips of as many rows as leave DW_WAVES waves, two a SIMD, where the level is
// large enough; below, strips down to one row high as long as there are no more
// than DW_ROW of them, from which on a strip's two rows of X beyond its own and its
// atomics cost more than its shorter chain gains: the least of a sweep of 64 to
// 320.  From DW_SPLIT strips of one row on, a wave takes all three tap rows.
// A gradient, us, split below 512 / 1024 / 2048 / 4096 / 8192 / 16384 such strips (and
// with the kernel of one tap a workgroup):
//   16 x 128                 412: 410 / 412 / 412 / 412 / 412 (420)
//   128 x 128                465: 462 / 462 / 460 / 462 / 463 (540)
//   200 x 256                555: 537 / 528 / 525 / 525 / 525 (720)
//   6 x 64 x 256             660: 652 / 637 / 621 / 626 / 623 (993)
//   8 x 128 x 256            853: 853 / 840 / 841 / 868 / 884 (1500)
//   16 x 256 x 256           1627: 1626 / 1626 / 1628 / 1643 / 1764 (3630)
constexpr long DW_WAVES = 2048, DW_ROW = 160, DW_SPLIT = 4096;

template <int CIN, int COUT, int TR>
void dw_launch(Net* n, int l, T4 X, T4 P, int nb, int rows, long lines) {
    const long waves = lines * ((P.H + rows - 1) / rows);
    hipLaunchKernelGGL((k_dw<CIN, COUT, TR>), dim3((unsigned)((waves + 3) / 4), 3 / TR), dim3(256), 0, n->stream, X, P,
                       n->g + n->woff[l], nb, rows);
}

template <int CIN, int COUT>
int dw(Net* n, int l, T4 X, T4 P, int nb) {
    const long lines = nb * (long)((P.W + 31) / 32) * DwSplit<CIN, COUT>::PAIRS;
    const long one = lines * P.H;  // strips one row high
    const int rows = (int)std::max(std::clamp(one / DW_ROW, 1l, 8l), one / DW_WAVES);
    if (one < DW_SPLIT)
        dw_launch<CIN, COUT, 1>(n, l, X, P, nb, rows, lines);
    else
        dw_launch<CIN, COUT, 3>(n, l, X, P, nb, rows, lines);
    SG_HIP(hipGetLastError());
    return SG_OK;
}

#define NN_TRY(x)               \
    do {                        \
        int _r = (x);           \
        if (_r) return _r;      \
    } while (0)

const bf16* WT(Net* n, int l) { return n->wt + n->woff[l]; }
const bf16* WF(Net* n, int l) { return n->wf + n->foff[l]; }

int refresh_bf16(Net* n) {
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks((long)n->nw)), dim3(256), 0, n->stream, (const float*)n->w, n->wt,
                       n->nw);
    for (int l = 1; l < NL; ++l) {
        const int cin = SPEC[l].cin, cout = SPEC[l].cout;
        hipLaunchKernelGGL(k_flip, dim3(blocks((long)cin * kpad(cout))), dim3(256), 0, n->stream,
                           (const bf16*)(n->wt + n->woff[l]), n->wf + n->foff[l], cin, cout);
    }
    SG_HIP(hipGetLastError());
    return SG_OK;
}

}  // namespace

size_t num_weights() {
    size_t s = 0;
    for (int l = 0; l < NL; ++l) s += (size_t)SPEC[l].cout * kpad(SPEC[l].cin);
    return s;
}

void destroy(Net* n) {
    for (void* p : n->allocs) (void)hipFree(p);
    n->allocs.clear();
}

int create(Net* n, int H, int W, int B, hipStream_t s) {
    if (H % 8 || W % 128 || H <= 0 || B <= 0) {
        set_error("learned warm start: the net needs H % 8 == 0 and W % 128 == 0");
        return SG_ERR_ARG;
    }
    n->H = H;
    n->W = W;
    n->B = B;
    n->stream = s;
    size_t o = 0, f = 0;
    for (int l = 0; l < NL; ++l) {
        n->woff[l] = o;
        n->foff[l] = f;
        o += (size_t)SPEC[l].cout * kpad(SPEC[l].cin);
        f += (size_t)SPEC[l].cin * kpad(SPEC[l].cout);
    }
    n->woff[NL] = o;
    n->foff[NL] = f;
    n->nw = o;
    auto alloc = [&](size_t bytes) -> void* {
        void* p = nullptr;
        if (hipMalloc(&p, bytes) != hipSuccess) return nullptr;
        if (hipMemset(p, 0, bytes) != hipSuccess) {
            (void)hipFree(p);
            return nullptr;
        }
        n->allocs.push_back(p);
        return p;
    };
    n->w = (float*)alloc(o * 4);
    n->g = (float*)alloc(o * 4);
    n->m = (float*)alloc(o * 4);
    n->v = (float*)alloc(o * 4);
    n->wt = (bf16*)alloc(o * 2);
    n->wf = (bf16*)alloc(f * 2);
    n->y = (float*)alloc((size_t)B * H * W * 4);
    n->loss = (float*)alloc(4);
    if (!n->w || !n->g || !n->m || !n->v || !n->wt || !n->wf || !n->y || !n->loss) {
        destroy(n);
        return SG_ERR_ALLOC;
    }
    bool ok = true;
    auto t4 = [&](int lvl, int C) {
        T4 t;
        t.H = H >> lvl;
        t.W = W >> lvl;
        t.C = C;
        t.p = (bf16*)alloc((size_t)B * (t.H + 2) * (t.W + 2) * C * 2);
        if (!t.p) ok = false;
        return t;
    };
    n->e0a = t4(0, 16); n->e0 = t4(0, 16); n->d1 = t4(1, 16);
    n->e1a = t4(1, 32); n->e1 = t4(1, 32); n->d2 = t4(2, 32);
    n->e2a = t4(2, 64); n->e2 = t4(2, 64); n->d3 = t4(3, 64);
    n->e3a = t4(3, 128); n->e3 = t4(3, 128);
    n->u2 = t4(2, 128); n->g2a = t4(2, 64); n->g2 = t4(2, 64);
    n->u1 = t4(1, 64); n->g1a = t4(1, 32); n->g1 = t4(1, 32);
    n->u0 = t4(0, 32); n->g0a = t4(0, 16); n->g0 = t4(0, 16);
    n->gout = t4(0, 16); n->P13 = t4(0, 16); n->P12 = t4(0, 16); n->du0 = t4(0, 32);
    n->P11 = t4(1, 32); n->P10 = t4(1, 32); n->du1 = t4(1, 64);
    n->P9 = t4(2, 64); n->P8 = t4(2, 64); n->du2 = t4(2, 128);
    n->P7 = t4(3, 128); n->P6 = t4(3, 128); n->dd3 = t4(3, 64);
    n->P5 = t4(2, 64); n->P4 = t4(2, 64); n->dd2 = t4(2, 32);
    n->P3 = t4(1, 32); n->P2 = t4(1, 32); n->dd1 = t4(1, 16);
    n->P1 = t4(0, 16); n->P0 = t4(0, 16);
    if (!ok) {
        destroy(n);
        return SG_ERR_ALLOC;
    }
    return SG_OK;
}

int set_weights(Net* n, const float* host) {
    SG_HIP(hipMemcpyAsync(n->w, host, n->nw * 4, hipMemcpyHostToDevice, n->stream));
    hipLaunchKernelGGL(k_fill, dim3(blocks((long)n->nw)), dim3(256), 0, n->stream, n->m, n->nw, 0.f);
    hipLaunchKernelGGL(k_fill, dim3(blocks((long)n->nw)), dim3(256), 0, n->stream, n->v, n->nw, 0.f);
    n->step = 0;
    NN_TRY(refresh_bf16(n));
    SG_HIP(hipStreamSynchronize(n->stream));
    return SG_OK;
}

int get_weights(Net* n, float* host) {
    SG_HIP(hipMemcpyAsync(host, n->w, n->nw * 4, hipMemcpyDeviceToHost, n->stream));
    SG_HIP(hipStreamSynchronize(n->stream));
    return SG_OK;
}

int forward(Net* n, const bf16* Xp, int nb) {
    if (nb < 1 || nb > n->B) {
        set_error("learned warm start: batch larger than the net's capacity");
        return SG_ERR_ARG;
    }
    T4 X;
    X.p = const_cast<bf16*>(Xp);
    X.H = n->H;
    X.W = n->W;
    X.C = CIN0;
    const T4 none;
    const hipStream_t s = n->stream;
    auto pool = [&](T4 a, T4 b) {
        hipLaunchKernelGGL(k_pool, dim3(blocks((long)nb * b.H * b.W * (b.C / 8))), dim3(256), 0, s, a, b, nb);
    };
    auto up = [&](T4 a, T4 b) {
        hipLaunchKernelGGL(k_up, dim3(blocks((long)nb * b.H * b.W * (b.C / 8))), dim3(256), 0, s, a, b, nb);
    };
    NN_TRY((conv<8, 16>(n, X, WT(n, 0), n->e0a, none, nullptr, nb, E_RELU)));
    NN_TRY((conv<16, 16>(n, n->e0a, WT(n, 1), n->e0, none, nullptr, nb, E_RELU)));
    pool(n->e0, n->d1);
    NN_TRY((conv<16, 32>(n, n->d1, WT(n, 2), n->e1a, none, nullptr, nb, E_RELU)));
    NN_TRY((conv<32, 32>(n, n->e1a, WT(n, 3), n->e1, none, nullptr, nb, E_RELU)));
    pool(n->e1, n->d2);
    NN_TRY((conv<32, 64>(n, n->d2, WT(n, 4), n->e2a, none, nullptr, nb, E_RELU)));
    NN_TRY((conv<64, 64>(n, n->e2a, WT(n, 5), n->e2, none, nullptr, nb, E_RELU)));
    pool(n->e2, n->d3);
    NN_TRY((conv<64, 128>(n, n->d3, WT(n, 6), n->e3a, none, nullptr, nb, E_RELU)));
    NN_TRY((conv<128, 128>(n, n->e3a, WT(n, 7), n->e3, none, nullptr, nb, E_RELU)));
    up(n->e3, n->u2);
    NN_TRY((conv<128, 64>(n, n->u2, WT(n, 8), n->g2a, n->e2, nullptr, nb, E_RELU_SKIP)));
    NN_TRY((conv<64, 64>(n, n->g2a, WT(n, 9), n->g2, none, nullptr, nb, E_RELU)));
    up(n->g2, n->u1);
    NN_TRY((conv<64, 32>(n, n->u1, WT(n, 10), n->g1a, n->e1, nullptr, nb, E_RELU_SKIP)));
    NN_TRY((conv<32, 32>(n, n->g1a, WT(n, 11), n->g1, none, nullptr, nb, E_RELU)));
    up(n->g1, n->u0);
    NN_TRY((conv<32, 16>(n, n->u0, WT(n, 12), n->g0a, n->e0, nullptr, nb, E_RELU_SKIP)));
    NN_TRY((conv<16, 16>(n, n->g0a, WT(n, 13), n->g0, none, nullptr, nb, E_RELU)));
    NN_TRY((conv<16, 16>(n, n->g0, WT(n, 14), none, none, n->y, nb, E_OUT)));
    SG_HIP(hipGetLastError());
    return SG_OK;
}

int backward(Net* n, const bf16* Xp, const float* t, const float* mask, int nb) {
    NN_TRY(forward(n, Xp, nb));
    T4 X;
    X.p = const_cast<bf16*>(Xp);
    X.H = n->H;
    X.W = n->W;
    X.C = CIN0;
    const T4 none;
    const hipStream_t s = n->stream;
    hipLaunchKernelGGL(k_fill, dim3(blocks((long)n->nw)), dim3(256), 0, s, n->g, n->nw, 0.f);
    hipLaunchKernelGGL(k_fill, dim3(1), dim3(256), 0, s, n->loss, (size_t)1, 0.f);
    const long npx = (long)nb * n->H * n->W;
    // a workgroup a CU before any takes more than its first 256 pixels
    const int per = (int)std::clamp(npx / (256 * 256), 1l, 8l);
    hipLaunchKernelGGL(k_loss, dim3((unsigned)((npx + 256 * per - 1) / (256 * per))), dim3(256), 0, s,
                       (const float*)n->y, t, mask, n->gout, nb, 1.f / (float)npx, per, n->loss);
    auto upT = [&](T4 d, T4 act, T4 P) {
        hipLaunchKernelGGL(k_upT_mask, dim3(blocks((long)nb * P.H * P.W * (P.C / 8))), dim3(256), 0, s, d, act, P,
                           nb);
    };
    auto poolT = [&](T4 dd, T4 skip, T4 act, T4 P) {
        hipLaunchKernelGGL(k_poolT_add_mask, dim3(blocks((long)nb * P.H * P.W * (P.C / 8))), dim3(256), 0, s, dd,
                           skip, act, P, nb);
    };
    NN_TRY((dw<16, 16>(n, 14, n->g0, n->gout, nb)));
    NN_TRY((conv<16, 16>(n, n->gout, WF(n, 14), n->P13, n->g0, nullptr, nb, E_MASK)));
    NN_TRY((dw<16, 16>(n, 13, n->g0a, n->P13, nb)));
    NN_TRY((conv<16, 16>(n, n->P13, WF(n, 13), n->P12, n->g0a, nullptr, nb, E_MASK)));
    NN_TRY((dw<32, 16>(n, 12, n->u0, n->P12, nb)));
    NN_TRY((conv<16, 32>(n, n->P12, WF(n, 12), n->du0, none, nullptr, nb, E_PLAIN)));
    upT(n->du0, n->g1, n->P11);
    NN_TRY((dw<32, 32>(n, 11, n->g1a, n->P11, nb)));
    NN_TRY((conv<32, 32>(n, n->P11, WF(n, 11), n->P10, n->g1a, nullptr, nb, E_MASK)));
    NN_TRY((dw<64, 32>(n, 10, n->u1, n->P10, nb)));
    NN_TRY((conv<32, 64>(n, n->P10, WF(n, 10), n->du1, none, nullptr, nb, E_PLAIN)));
    upT(n->du1, n->g2, n->P9);
    NN_TRY((dw<64, 64>(n, 9, n->g2a, n->P9, nb)));
    NN_TRY((conv<64, 64>(n, n->P9, WF(n, 9), n->P8, n->g2a, nullptr, nb, E_MASK)));
    NN_TRY((dw<128, 64>(n, 8, n->u2, n->P8, nb)));
    NN_TRY((conv<64, 128>(n, n->P8, WF(n, 8), n->du2, none, nullptr, nb, E_PLAIN)));
    upT(n->du2, n->e3, n->P7);
    NN_TRY((dw<128, 128>(n, 7, n->e3a, n->P7, nb)));
    NN_TRY((conv<128, 128>(n, n->P7, WF(n, 7), n->P6, n->e3a, nullptr, nb, E_MASK)));
    NN_TRY((dw<64, 128>(n, 6, n->d3, n->P6, nb)));
    NN_TRY((conv<128, 64>(n, n->P6, WF(n, 6), n->dd3, none, nullptr, nb, E_PLAIN)));
    poolT(n->dd3, n->P8, n->e2, n->P5);
    NN_TRY((dw<64, 64>(n, 5, n->e2a, n->P5, nb)));
    NN_TRY((conv<64, 64>(n, n->P5, WF(n, 5), n->P4, n->e2a, nullptr, nb, E_MASK)));
    NN_TRY((dw<32, 64>(n, 4, n->d2, n->P4, nb)));
    NN_TRY((conv<64, 32>(n, n->P4, WF(n, 4), n->dd2, none, nullptr, nb, E_PLAIN)));
    poolT(n->dd2, n->P10, n->e1, n->P3);
    NN_TRY((dw<32, 32>(n, 3, n->e1a, n->P3, nb)));
    NN_TRY((conv<32, 32>(n, n->P3, WF(n, 3), n->P2, n->e1a, nullptr, nb, E_MASK)));
    NN_TRY((dw<16, 32>(n, 2, n->d1, n->P2, nb)));
    NN_TRY((conv<32, 16>(n, n->P2, WF(n, 2), n->dd1, none, nullptr, nb, E_PLAIN)));
    poolT(n->dd1, n->P12, n->e0, n->P1);
    NN_TRY((dw<16, 16>(n, 1, n->e0a, n->P1, nb)));
    NN_TRY((conv<16, 16>(n, n->P1, WF(n, 1), n->P0, n->e0a, nullptr, nb, E_MASK)));
    NN_TRY((dw<8, 16>(n, 0, X, n->P0, nb)));
    SG_HIP(hipGetLastError());
    return SG_OK;
}

int adam_step(Net* n, float lr) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    n->step += 1;
    const float c1 = 1.f / (1.f - powf(b1, (float)n->step));
    const float c2 = 1.f / (1.f - powf(b2, (float)n->step));
    hipLaunchKernelGGL(k_adam, dim3(blocks((long)n->nw)), dim3(256), 0, n->stream, n->w, (const float*)n->g, n->m,
                       n->v, n->nw, lr, b1, b2, c1, c2, eps);
    SG_HIP(hipGetLastError());
    return refresh_bf16(n);
}

}  // namespace nn
}  // namespace sg
