// unet.hip - the warm-start network's training and inference kernels (gfx950).
//
// Activations are BF16, NHWC (channels contiguous), with every channel count
// a multiple of 32; weights of a 3x3 convolution are [9][Cout][Cin] (tap =
// 3*(dy+1) + (dx+1)); accumulation is FP32 on the matrix cores
// (v_mfma_f32_16x16x32_bf16); activation gradients are FP32.  Rounding to
// BF16 is round-to-nearest-even, written out (f2bf), so the CPU oracle can
// reproduce every rounding point.
//
// 3x3 convolution = implicit GEMM: M = pixels, N = output channels, K = 9 x
// Cin.  A wave owns 64 pixels (4 MFMA row blocks) x 16*NJ channels, so each
// weight fragment is reused by 4 MFMAs from registers and each input
// fragment by NJ; the K loop walks the 9 taps x 32-channel chunks with 16-byte
// loads (zero outside the image).  The data gradient is the same kernel run
// on the flipped, transposed weights; the weight gradient is a split-K GEMM
// over pixels through LDS-transposed tiles with a fixed-order reduction
// (deterministic, no atomics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <type_traits>

#include "glide_unet.h"

namespace glide {
int set_error(int code, const char *msg);
}

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t bf16_t;

int ufail(int code, const std::string &msg) { return glide::set_error(code, msg.c_str()); }
int ucheck(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return ufail((int)e, std::string(what) + ": " + hipGetErrorString(e));
    return GLIDE_OK;
}

}  // namespace

__device__ __forceinline__ float bf2f(bf16_t h)
{
    uint32_t u = (uint32_t)h << 16;
    float f;
    __builtin_memcpy(&f, &u, 4);
    return f;
}
// round to nearest even (NaN stays NaN)
__device__ __forceinline__ bf16_t f2bf(float f)
{
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x40);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
}

union Frag {
    uint4 raw;
    bf16x8 v;
};
// 8 channels in one 16-byte access
union Bf8 {
    uint4 raw;
    bf16_t h[8];
};

// ---------------------------------------------------------------------------
// 3x3 convolution, implicit GEMM on MFMA.
// MODE 0 (forward): out_bf16[p][co] = act(bias[co] + sum_{t,ci} W[t][co][ci] x[p+off_t][ci])
//        x = concat(xa (CA ch), xb (CB ch)); act = ReLU when relu != 0.
// MODE 1 (data gradient): the same sum without bias/act into FP32 outputs split
//        by channel: co < SA -> ga[p][co] (+)= ..., else gb[p][co - SA] (+)= ...
// MODE 2 (data gradient through the input's ReLU): out_bf16[p][co] =
//        bf16(ya[p][co] > 0 ? sum : 0), what MODE 1 followed by the ReLU's
//        backward gives without the FP32 gradient's round trip through memory.
//
// A workgroup of NW waves owns 2 NW rows x 32 columns of one image x 32 output
// channels: it stages the (2 NW + 2) x 34 input pixels of every channel (NCH
// chunks of 32) in LDS once (zero outside the image), so the nine taps read
// memory once, and a wave takes 2 rows (4 MFMA blocks of 16 pixels).  An LDS
// pixel is 32 channels in 64 bytes, its four 16-byte pieces swapped by its
// column / 4, which puts the reads of 16 consecutive pixels in different banks.  Weight fragments come from the
// caches, three steps ahead.  The weights are the MFMA's row operand, in an
// order that leaves a lane with 8 consecutive output channels of its pixel:
// one 16-byte store (two for FP32) instead of 8 of 2 bytes.  The K loop walks
// the 9 taps x 32-channel chunks in that order whatever the tile, so the sums'
// bits do not depend on it.
//
// Balance per step: a wave issues 4 LDS reads and 2 weight loads of 1 KB for 8
// MFMAs of 16 cycles, about what LDS and L1 deliver to four waves in that
// time.  Reading the pixels of every tap from the caches and storing 2 bytes
// at a time took 30 us for 512^2 pixels of 32 -> 32 channels; this takes 13 us
// (7 us at the rate of a large copy).
// ---------------------------------------------------------------------------
constexpr int CV_W = 32;      // tile columns
constexpr int CV_LD = 32;     // LDS pitch of a pixel's 32 channels (bf16)

// f2bf without the NaN case (a NaN becomes some other value)
__device__ __forceinline__ uint32_t f2bf_num(float f)
{
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// 16-byte pieces a thread stages per round: all of them where that is at most 12 (18 for 6 chunks) loads in flight
constexpr int conv_round(int ne, int nch)
{
    const int most = (nch > 4 ? 18 : 12) / nch, rounds = (ne + most - 1) / most;
    return (ne + rounds - 1) / rounds;
}

constexpr size_t conv_lds(int nw, int nch) { return (size_t)nch * (2 * nw + 2) * (CV_W + 2) * CV_LD * sizeof(bf16_t); }
constexpr size_t conv_wlds(int ng, int nch) { return (size_t)9 * nch * 32 * ng * CV_LD * sizeof(bf16_t); }
// the weights go through LDS too where waves share them and a CU's 160 KB hold both
constexpr bool conv_wl(int nw, int ng, int nch) { return nw == 4 && conv_lds(nw, nch) + conv_wlds(ng, nch) <= 160 * 1024; }

template <int NW, int NG, int NCH, int MODE>
__global__ __launch_bounds__(64 * NW * NG, NCH == 1 ? 5 : NCH == 6 ? 2 : NCH == 3 ? 3 : 4) void k_conv3x3(const bf16_t *__restrict__ xa, int CA, int up,
                                                     const bf16_t *__restrict__ xb, int H, int W, int tiles_x,
                                                     int tiles, const bf16_t *__restrict__ Wt, int Cout,
                                                     const float *__restrict__ bias, int relu,
                                                     const bf16_t *__restrict__ ya, bf16_t *__restrict__ out,
                                                     bf16_t *__restrict__ pool,
                                                     float *__restrict__ ga, int SA, int acc_a,
                                                     float *__restrict__ gb, int acc_b)
{
    constexpr int PW = CV_W + 2, NPX = (2 * NW + 2) * PW, Cin = 32 * NCH;
    constexpr bool WL = conv_wl(NW, NG, NCH);
    __shared__ bf16_t sm[NCH * NPX * CV_LD];   // [chunk][pixel][CV_LD]
    __shared__ bf16_t smw[WL ? 9 * NCH * 32 * NG * CV_LD : 1];   // [tap][chunk][output channel][CV_LD]
    constexpr int NT = 64 * NW * NG;
    const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) % NW;
    const int r16 = lane & 15, kq = lane >> 4;   // fragment row / k-quarter
    const int n = blockIdx.x / tiles, tl = blockIdx.x - n * tiles;
    const int y0 = (tl / tiles_x) * 2 * NW, x0 = (tl % tiles_x) * CV_W;
    const int co0 = (blockIdx.y * NG + (tid >> 6) / NW) * 32;
    const long img = (long)n * H * W;

    // weight fragments of step (t, c): row m of fragment j is channel co0 + 8 (m / 4) + 4 j + m % 4
    const uint32_t wlane = ((co0 + 8 * (r16 >> 2) + (r16 & 3)) * Cin + 8 * kq) * 2u;
    const long tap = (long)Cout * Cin * 2;
    auto wload = [&](int t, int c, Frag(&B)[2]) {
        const char *b = (const char *)Wt + t * tap + 64 * c;
        B[0].raw = *(const uint4 *)(b + wlane);
        B[1].raw = *(const uint4 *)(b + 8 * Cin + wlane);
    };
    constexpr int D = NCH == 1 ? 3 : NCH == 3 ? 9 : 6;   // steps ahead, a divisor of the 3 NCH steps of a row of taps
    Frag B[D][2];
    if (!WL) {
#pragma unroll
        for (int s = 0; s < D; s++) wload(s / NCH, s % NCH, B[s]);
    }
    // staged weights: a tap's rows of this workgroup's channels are one block of memory
    constexpr int NWP = 9 * NCH * 128 * NG, NWE = WL ? (NWP + NT - 1) / NT : 1;
    uint4 wv[NWE];
    if (WL) {
#pragma unroll
        for (int k = 0; k < NWE; k++) {
            const int e = tid + NT * k, t = e / (NCH * 128 * NG), r = e - t * (NCH * 128 * NG);
            wv[k] = e < NWP ? *(const uint4 *)((const char *)Wt + t * tap + (long)blockIdx.y * (NCH * 2048 * NG) + 16 * r)
                            : uint4{0u, 0u, 0u, 0u};
        }
    }

    // The weights are not in the L2s when a layer starts, and the workgroups of an XCD walk them in step, each prefetch
    // a miss: so every XCD's workgroups first touch them, up to two lines of 128 bytes a thread (with few workgroups
    // the last of the weights stay untouched)
    uint32_t touched = 0;
    if (!WL) {
        const long lines = (9 * tap + 127) / 128;
        const unsigned b = blockIdx.x + gridDim.x * blockIdx.y, nb = (gridDim.x * gridDim.y + 7) / 8;
        const long l = (long)(b / 8) * NT + tid;
        if (l < lines) touched = *(const uint32_t *)((const char *)Wt + 128 * l);
        if (l + (long)nb * NT < lines) touched ^= *(const uint32_t *)((const char *)Wt + 128 * (l + (long)nb * NT));
    }
    // stage the input: 16-byte pieces, 4 per pixel and chunk
    constexpr int NE = (NPX * 4 + NT - 1) / NT, NB = conv_round(NE, NCH);   // pieces per thread, in flight x NCH
    const int CB = Cin - CA, ncha = CA / 32;
#pragma unroll
    for (int e0 = 0; e0 < NE; e0 += NB) {
        uint4 v[NB][NCH];
#pragma unroll
        for (int k = 0; k < NB; k++) {
            const int e = tid + NT * (e0 + k), px = e >> 2, q = e & 3;
            const int ry = px / PW, rx = px - ry * PW;
            const int y = y0 - 1 + ry, x = x0 - 1 + rx;
            const bool ok = e < NPX * 4 && y >= 0 && y < H && x >= 0 && x < W;
            const long p = img + (long)y * W + x;
            // xa at half the resolution: its pixel under this one
            const long pa = MODE == 0 && up ? ((long)n * (H / 2) + (y >> 1)) * (W / 2) + (x >> 1) : p;
            const bf16_t *a = xa + pa * CA + 8 * q, *b = xb + p * CB + 8 * q;
#pragma unroll
            for (int c = 0; c < NCH; c++)
                v[k][c] = ok ? *(const uint4 *)(c < ncha ? a + 32 * c : b + 32 * (c - ncha)) : uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int k = 0; k < NB; k++) {
            const int e = tid + NT * (e0 + k);
            if (e < NPX * 4) {
                const int px = e >> 2, lds = px * CV_LD + 8 * ((e & 3) ^ ((px % PW) >> 2 & 3));
#pragma unroll
                for (int c = 0; c < NCH; c++) *(uint4 *)(sm + c * NPX * CV_LD + lds) = v[k][c];
            }
        }
    }
    if (WL) {
#pragma unroll
        for (int k = 0; k < NWE; k++) {
            const int e = tid + NT * k, t = e / (NCH * 128 * NG), r = e - t * (NCH * 128 * NG);
            const int row = r / (4 * NCH), c = r % (4 * NCH) >> 2, q = r & 3;
            if (e < NWP) *(uint4 *)(smw + ((t * NCH + c) * 32 * NG + row) * CV_LD + 8 * (q ^ (row >> 3 & 3))) = wv[k];
        }
    }
    if (!WL) asm volatile("" ::"v"(touched));
    __syncthreads();

    f32x4 acc[4][2];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[a][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // pixel block a: row 2 wave + a / 2, columns 16 (a % 2) + r16; per column offset of the taps its swizzled address
    const bf16_t *base[3];
#pragma unroll
    for (int dx = 0; dx < 3; dx++)
        base[dx] = sm + (2 * wave * PW + r16 + dx) * CV_LD + 8 * (kq ^ ((r16 + dx) >> 2 & 3));
    auto aload = [&](int s, Frag(&A)[4]) {   // step s of a row of taps: tap s / NCH, chunk s % NCH
#pragma unroll
        for (int a = 0; a < 4; a++)
            A[a].raw = *(const uint4 *)(base[s / NCH] + (s % NCH * NPX + (a >> 1) * PW + 16 * (a & 1)) * CV_LD);
    };
    const bf16_t *wbase = smw + (32 * ((tid >> 6) / NW) + 8 * (r16 >> 2) + (r16 & 3)) * CV_LD + 8 * (kq ^ (r16 >> 2));
    auto bload = [&](int s, Frag(&b)[2]) {
        const bf16_t *w = wbase + s * 32 * NG * CV_LD;
        b[0].raw = *(const uint4 *)w;
        b[1].raw = *(const uint4 *)(w + 4 * CV_LD);
    };
    // with more channels fewer waves fit: the pixels of the next step load ahead (NA a divisor of a row's 3 NCH steps)
    constexpr int NA = NCH == 1 ? 1 : NCH == 3 ? 3 : 2;
    Frag A[NA][4];
    Frag Bl[NA][2];
    if (NA > 1) {
        aload(0, A[0]);
        if (WL) bload(0, Bl[0]);
    }
#pragma unroll 1
    for (int dy = 0; dy < 3; dy++) {
#pragma unroll
        for (int s = 0; s < 3 * NCH; s++) {   // step 3 NCH dy + s: tap 3 dy + s / NCH, chunk s % NCH
            constexpr int S = 3 * NCH;
            if (NA == 1) {
                aload(s, A[0]);
                if (WL) bload(s, Bl[0]);
            }
            if (NA > 1 && s + 1 < S) {
                aload(s + 1, A[(s + 1) % NA]);
                if (WL) bload(s + 1, Bl[(s + 1) % NA]);
            }
            if (NA > 1 && s + 1 == S) {   // past the last row: the last row again
#pragma unroll
                for (int dx = 0; dx < 3; dx++) base[dx] += dy < 2 ? PW * CV_LD : 0;
                wbase += dy < 2 ? S * 32 * NG * CV_LD : 0;
                aload(0, A[0]);
                if (WL) bload(0, Bl[0]);
            }
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int a = 0; a < 4; a++)
                    acc[a][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(WL ? Bl[s % NA][j].v : B[s % D][j].v, A[s % NA][a].v,
                                                                        acc[a][j], 0, 0, 0);
            if (WL) continue;
            const int q = s + D;   // past the last step: the last tap again
            const int t = 3 * dy + q / NCH;
            wload(t < 9 ? t : 8, q % NCH, B[s % D]);
        }
        if (NA == 1) {
#pragma unroll
            for (int dx = 0; dx < 3; dx++) base[dx] += PW * CV_LD;
            wbase += 3 * NCH * 32 * NG * CV_LD;
        }
    }

    // D fragment: row 4*kq + i of fragment j = channel co0 + 8*kq + 4*j + i, column r16 = pixel
    const int co = co0 + 8 * kq;
    float bs[8] = {};
    if (MODE == 0) {
        const float4 b0 = *(const float4 *)(bias + co), b1 = *(const float4 *)(bias + co + 4);
        bs[0] = b0.x, bs[1] = b0.y, bs[2] = b0.z, bs[3] = b0.w, bs[4] = b1.x, bs[5] = b1.y, bs[6] = b1.z, bs[7] = b1.w;
    }
    uint4 o4[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
        const int y = y0 + 2 * wave + (a >> 1), x = x0 + 16 * (a & 1) + r16;
        o4[a] = uint4{0u, 0u, 0u, 0u};
        if (y >= H || x >= W) continue;
        const long p = img + (long)y * W + x;
        if (MODE != 1) {
            uint32_t h[8];
            Bf8 y8;
            if (MODE == 2) y8.raw = *(const uint4 *)(ya + p * Cout + co);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float val = acc[a][i >> 2][i & 3] + bs[i];
                if (MODE == 0)
                    h[i] = relu ? f2bf_num(fmaxf(val, 0.0f)) : (uint32_t)f2bf(val);   // fmaxf leaves no NaN
                else
                    h[i] = f2bf(bf2f(y8.h[i]) > 0.0f ? acc[a][i >> 2][i & 3] : 0.0f);
            }
            o4[a] = uint4{h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16};
            *(uint4 *)(out + p * Cout + co) = o4[a];
        } else {
            const bool first = co0 < SA;   // 32-channel groups lie in one of the outputs
            float4 *d = (float4 *)(first ? ga + p * SA + co : gb + p * (Cout - SA) + (co - SA));
            float4 v0 = {acc[a][0][0], acc[a][0][1], acc[a][0][2], acc[a][0][3]};
            float4 v1 = {acc[a][1][0], acc[a][1][1], acc[a][1][2], acc[a][1][3]};
            if (first ? acc_a : acc_b) {
                const float4 o0 = d[0], o1 = d[1];
                v0 = float4{o0.x + v0.x, o0.y + v0.y, o0.z + v0.z, o0.w + v0.w};
                v1 = float4{o1.x + v1.x, o1.y + v1.y, o1.z + v1.z, o1.w + v1.w};
            }
            d[0] = v0;
            d[1] = v1;
        }
    }
    // 2x2 mean of the output as k_pool2 forms it: the lane's two rows and the next lane's (H and W even)
    if (MODE == 0 && pool) {
#pragma unroll
        for (int a = 0; a < 2; a++) {
            Bf8 q0, q1, q2, q3, o;
            q0.raw = o4[a];
            q2.raw = o4[a + 2];
            auto next = [](uint4 v) {
                return uint4{(uint32_t)__shfl_xor((int)v.x, 1), (uint32_t)__shfl_xor((int)v.y, 1),
                             (uint32_t)__shfl_xor((int)v.z, 1), (uint32_t)__shfl_xor((int)v.w, 1)};
            };
            q1.raw = next(q0.raw);
            q3.raw = next(q2.raw);
            const int y = y0 + 2 * wave, x = x0 + 16 * a + r16;
            if (y >= H || x >= W || (r16 & 1)) continue;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float s = ((bf2f(q0.h[i]) + bf2f(q1.h[i])) + bf2f(q2.h[i])) + bf2f(q3.h[i]);
                o.h[i] = f2bf(0.25f * s);
            }
            *(uint4 *)(pool + (((long)n * (H / 2) + y / 2) * (W / 2) + x / 2) * Cout + co) = o.raw;
        }
    }
}

// The same convolution reading every tap's pixels from the caches, for input
// channel counts that k_conv3x3 has no instance for (160, and above 192, whose
// halo tile outgrows its LDS): a wave owns 64 consecutive pixels x 16 NJ
// channels.  Grid: x = pixel blocks of 256 (4
// waves x 64), y = output-channel groups of 16 NJ.  The same sums, bit for bit.
// UP (xa at half the resolution) is an instance of its own: as an argument its
// shifts cost every convolution 5 to 9% (160 -> 64 channels of 128^2: 37.6 -> 34.8 us).
template <int NJ, int MODE, bool UP>
__global__ __launch_bounds__(256) void k_conv3x3_direct(const bf16_t *__restrict__ xa, int CA,
                                                        const bf16_t *__restrict__ xb,
                                                        int CB, int N, int H, int W, const bf16_t *__restrict__ Wt, int Cout,
                                                        const float *__restrict__ bias, int relu, const bf16_t *__restrict__ ya,
                                                        bf16_t *__restrict__ out,
                                                        float *__restrict__ ga, int SA, int acc_a, float *__restrict__ gb,
                                                        int acc_b)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int Cin = CA + CB;
    const long P = (long)N * H * W;
    const long pbase = (long)blockIdx.x * 256 + wave * 64;
    const int co0 = blockIdx.y * 16 * NJ;
    const int r16 = lane & 15, kq = lane >> 4;   // fragment row / k-quarter
    // the 4 pixels this lane feeds as A rows
    int py[4], px[4], pn[4];
    bool pv[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
        long p = pbase + 16 * a + r16;
        pv[a] = p < P;
        long q = pv[a] ? p : 0;
        px[a] = (int)(q % W);
        long t = q / W;
        py[a] = (int)(t % H);
        pn[a] = (int)(t / H);
    }
    f32x4 acc[4][NJ];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[a][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // K steps s = (tap t, 32-channel chunk c): fragments of step s + 1 are
    // loaded while the MFMAs of step s run (the accumulation order over s is
    // the plain tap-major, channel-minor order)
    const int nch = Cin / 32, nsteps = 9 * nch;
    auto load = [&](int s, Frag(&A)[4], Frag(&B)[NJ]) {
        const int t = s / nch, c0 = (s - t * nch) * 32;
        const int dy = t / 3 - 1, dx = t % 3 - 1;
        const bf16_t *xs = c0 < CA ? xa : xb;
        const int cs = c0 < CA ? CA : CB, cc = (c0 < CA ? c0 : c0 - CA) + 8 * kq;
#pragma unroll
        for (int a = 0; a < 4; a++) {
            const int y = py[a] + dy, x = px[a] + dx;
            const bool ok = pv[a] && y >= 0 && y < H && x >= 0 && x < W;
            const int h = UP && c0 < CA;   // xa at half the resolution
            const long src = ok ? (((long)pn[a] * (H >> h) + (y >> h)) * (W >> h) + (x >> h)) : 0;
            A[a].raw = ok ? *(const uint4 *)(xs + src * cs + cc) : uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int j = 0; j < NJ; j++)
            B[j].raw = *(const uint4 *)(Wt + ((long)t * Cout + co0 + 16 * j + r16) * Cin + c0 + 8 * kq);
    };
    auto mma = [&](const Frag(&A)[4], const Frag(&B)[NJ]) {
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int a = 0; a < 4; a++)
                acc[a][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[a].v, B[j].v, acc[a][j], 0, 0, 0);
    };
    Frag Ac[4], Bc[NJ], An[4], Bn[NJ];
    load(0, Ac, Bc);
#pragma unroll 1
    for (int s = 0; s < nsteps; s++) {
        if (s + 1 < nsteps) load(s + 1, An, Bn);
        mma(Ac, Bc);
#pragma unroll
        for (int a = 0; a < 4; a++) Ac[a] = An[a];
#pragma unroll
        for (int j = 0; j < NJ; j++) Bc[j] = Bn[j];
    }
    // D fragment: row (pixel) = 4*kq + i, column (channel) = r16
#pragma unroll
    for (int a = 0; a < 4; a++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const long p = pbase + 16 * a + 4 * kq + i;
            if (p >= P) continue;
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                const int co = co0 + 16 * j + r16;
                float val = acc[a][j][i];
                if (MODE == 0) {
                    val += bias[co];
                    if (relu) val = fmaxf(val, 0.0f);
                    out[p * Cout + co] = f2bf(val);
                } else if (MODE == 2) {
                    out[p * Cout + co] = f2bf(bf2f(ya[p * Cout + co]) > 0.0f ? val : 0.0f);
                } else {
                    if (co < SA) {
                        float *d = ga + p * SA + co;
                        *d = acc_a ? *d + val : val;
                    } else {
                        float *d = gb + p * (Cout - SA) + (co - SA);
                        *d = acc_b ? *d + val : val;
                    }
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Weight gradient: partial[z][t][co][ci] = sum over the z-th pixel chunk of
// dz[p][co] * x[p + off_t][ci]; one block = 32 co x 32 ci of all nine taps.
//
// A GEMM with K = pixels, whose operands lie channel-contiguous in memory: the
// block stages WG_PX pixels of dz and of the three image rows of x around them
// in LDS as they lie (16-byte stores), and ds_read_b64_tr_b16 hands each lane
// the four consecutive pixels of its channel that a fragment needs.  A tap's
// column shift is a row offset into the staged pixels, so x is read from
// memory once for its nine taps.  Waves 0 to 2 take the three taps of image
// row w - 1: per 32 pixels they read 2 dz and 6 x fragments for 12 MFMAs.
// Wave 3 stages dz and, in the blocks of the first 32 input channels, adds up
// the bias gradient from the same staged pixels, which costs no time beside
// the MFMA waves.  The pitch of 96 bytes puts the four pixels that 16 lanes read in
// different banks.  Every (tap, co, ci) sums its chunk in steps of 32 pixels in
// pixel order, and every channel's bias gradient pixel by pixel, so the bits
// depend on neither the tile nor the grid.
//
// A block is a serial chain of chunk / WG_PX tiles (often one block per CU), so
// what counts is the time of one tile: loads run two tiles ahead, and a tile
// whose pixels all lie inside the image (most of them) loads without tests.
// For a 16 x 256^2 training step's 13 layers: 5.0 ms with one tap per block and
// 2-byte transposing stores (and 0.64 ms for the bias gradients by themselves),
// 1.1 ms with loads one tile ahead and tested addresses, 0.72 ms now.
// ---------------------------------------------------------------------------
constexpr int WG_PX = 128;   // pixels per staged tile
constexpr int WG_LD = 48;    // LDS pitch of a pixel's 32 channels (bf16)
constexpr int WG_NR = WG_PX / 16 + 1;   // 16-byte pieces of a staged row per lane

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// rows 0-3 and 4-7 (pitch WG_LD) from t of one channel per lane, in row order;
// t: the lane's row (lane % 16 / 4) and 4-channel group (lane % 4) of its 16 channels
__device__ __forceinline__ Frag tr_frag(const bf16_t *t)
{
    union {
        s16x4 h[2];
        Frag f;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)t);
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(t + 4 * WG_LD));
    return u.f;
}

__global__ __launch_bounds__(256, 2) void k_conv3x3_wgrad(const bf16_t *__restrict__ dz, int Cout,
                                                          const bf16_t *__restrict__ xa, int CA,
                                                          const bf16_t *__restrict__ xb, int CB, int N, int H, int W,
                                                          long chunk, float *__restrict__ partial,
                                                          float *__restrict__ part_b)
{
    __shared__ bf16_t sD[WG_PX][WG_LD];          // dz of pixel p0 + k
    __shared__ bf16_t sX[3][WG_PX + 2][WG_LD];   // x of pixel p0 - 1 + k, image row dy = -1, 0, 1
    const int Cin = CA + CB;
    const int ci0 = blockIdx.x * 32, co0 = blockIdx.y * 32;
    const long P = (long)N * H * W, HW = (long)H * W;
    const long p_lo = (long)blockIdx.z * chunk, p_hi = p_lo + chunk < P ? p_lo + chunk : P;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), dy = w - 1;
    const int r16 = lane & 15, kq = lane >> 4;
    const bool is_x = w < 3;
    // the row that this wave stages: element k is pixel p0 + shift + k of src
    const bf16_t *src = is_x ? (ci0 < CA ? xa + ci0 : xb + (ci0 - CA)) : dz + co0;
    const int cs = is_x ? (ci0 < CA ? CA : CB) : Cout;
    const long shift = is_x ? (long)dy * W - 1 : 0;
    const int len = is_x ? WG_PX + 2 : WG_PX;
    bf16_t(*row)[WG_LD] = is_x ? sX[w] : sD;
    const int s0 = lane >> 2;
    const bf16_t *lsrc = src + (long)s0 * cs + 8 * (lane & 3);
    // position in its image of the x row's first pixel; the rows above (dy = -1)
    // and below (dy = 1) the image are zero
    const bool in32 = P + 2 * HW < (1L << 31);   // a 64-bit remainder is a tenth of the time of a call of few pixels
    long r0 = p_lo + shift + 2 * HW;   // shift >= -HW - 1
    r0 = !is_x ? 0 : in32 ? (long)((uint32_t)r0 % (uint32_t)HW) : r0 % HW;
    const long bad_lo = dy < 0 ? HW - W : 0, bad_hi = dy == 0 ? 0 : bad_lo + W;
    // k % HW for k < HW + 16 WG_NR; an image smaller than a staged row by its reciprocal (subtracting it again and
    // again took 300 images of one pixel from 15 to 88 us)
    const uint32_t inv = HW < 16 * WG_NR ? (uint32_t)((65535 + HW) / HW) : 0;   // exact: k (HW inv - 2^16) < 2^16
    auto wrap = [&](long k) { return inv ? k - HW * (long)(((uint32_t)k * inv) >> 16) : (k >= HW ? k - HW : k); };
    auto load = [&](long p0, uint4(&r)[WG_NR]) {
        const long q0 = p0 + shift;
        const bool inside = is_x ? q0 >= 0 && q0 + len <= P && r0 + len <= HW && (r0 + len <= bad_lo || r0 >= bad_hi)
                                 : q0 + len <= p_hi;
        const bf16_t *b = lsrc + q0 * cs;
        if (inside) {
#pragma unroll
            for (int m = 0; m < WG_NR; m++)
                if (16 * m + s0 < len) r[m] = *(const uint4 *)(b + 16 * m * cs);
        } else {
#pragma unroll
            for (int m = 0; m < WG_NR; m++) {
                const int s = s0 + 16 * m;
                const long q = q0 + s;
                bool ok = s < len && q >= 0 && q < (is_x ? P : p_hi);
                if (is_x) {
                    const long k = wrap(r0 + s);
                    ok = ok && !(k >= bad_lo && k < bad_hi);
                }
                r[m] = ok ? *(const uint4 *)(b + 16 * m * cs) : uint4{0u, 0u, 0u, 0u};
            }
        }
        if (is_x) r0 = wrap(r0 + WG_PX);
    };
    f32x4 acc[3][2][2];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++) acc[d][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum = 0.0f;
    // column of the lane's first pixel (8 kq past the step's first)
    int col = in32 ? (int)((uint32_t)(p_lo + 8 * kq) % (uint32_t)W) : (int)((p_lo + 8 * kq) % W);
    const int cstep = 32 % W;
    // the lane's corner of a fragment at step 0: pixel 8 kq + r16 / 4, channels 4 (r16 % 4)
    const int fo = (8 * kq + (r16 >> 2)) * WG_LD + 4 * (r16 & 3);
    const bf16_t *xrow = &sX[is_x ? w : 0][0][0];
    auto step = [&](long p0, int st, auto plain) {
        const int o = fo + 32 * st * WG_LD;
        Frag A[2], B[3][2];
#pragma unroll
        for (int a = 0; a < 2; a++) A[a] = tr_frag(&sD[0][0] + o + 16 * a);
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int b = 0; b < 2; b++) B[d][b] = tr_frag(xrow + o + d * WG_LD + 16 * b);
        // x is 0 left of column 0 (tap dx = -1) and right of column W - 1 (dx = 1)
        if (plain) {
            const uint32_t ml = col == 0 ? 0xffff0000u : 0xffffffffu, mr = col == W - 8 ? 0x0000ffffu : 0xffffffffu;
#pragma unroll
            for (int b = 0; b < 2; b++) {
                B[0][b].raw.x &= ml;
                B[2][b].raw.w &= mr;
            }
        } else {
            uint32_t m[3][4] = {};
            int c = col;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const uint32_t h = p0 + 32 * st + 8 * kq + e < p_hi ? 0xffffu << (16 * (e & 1)) : 0u;
                m[0][e >> 1] |= c > 0 ? h : 0u;
                m[1][e >> 1] |= h;
                m[2][e >> 1] |= c < W - 1 ? h : 0u;
                c = c + 1 == W ? 0 : c + 1;
            }
#pragma unroll
            for (int d = 0; d < 3; d++)
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    B[d][b].raw.x &= m[d][0];
                    B[d][b].raw.y &= m[d][1];
                    B[d][b].raw.z &= m[d][2];
                    B[d][b].raw.w &= m[d][3];
                }
        }
        col += cstep;
        col = col >= W ? col - W : col;
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < 2; b++)
                    acc[d][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[a].v, B[d][b].v, acc[d][a][b], 0, 0, 0);
    };
    // lanes 0-31: bias gradient of channel co0 + lane, four pixels per read
    const bool do_b = part_b && blockIdx.x == 0 && lane < 32;
    const bf16_t *bcol = &sD[r16 >> 2][16 * (kq & 1) + 4 * (r16 & 3)];
    auto tile = [&](long p0, uint4(&r)[WG_NR]) {
        __syncthreads();   // the previous tile has been read
#pragma unroll
        for (int m = 0; m < WG_NR; m++)
            if (16 * m + s0 < len) *(uint4 *)&row[16 * m + s0][8 * (lane & 3)] = r[m];
        __syncthreads();
        if (p0 + 2 * WG_PX < p_hi) load(p0 + 2 * WG_PX, r);
        if (is_x) {
            // 8 consecutive pixels lie in one image row where W % 8 == 0 (chunks start at multiples of 8)
            if ((W & 7) == 0 && p0 + WG_PX <= p_hi) {
#pragma unroll
                for (int st = 0; st < WG_PX / 32; st++) step(p0, st, std::true_type{});
            } else {
#pragma unroll 1
                for (int st = 0; st < WG_PX / 32 && p0 + 32 * st < p_hi; st++) step(p0, st, std::false_type{});
            }
        } else if (do_b) {
            const int n = p_hi - p0 < WG_PX ? (int)(p_hi - p0) : WG_PX;
            if (n == WG_PX) {
#pragma unroll 8
                for (int k = 0; k < WG_PX; k += 4) {
                    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(bcol + k * WG_LD));
#pragma unroll
                    for (int e = 0; e < 4; e++) bsum += bf2f((bf16_t)v[e]);
                }
            } else {
                for (int k = 0; k < n; k++) bsum += bf2f(sD[k][lane]);
            }
        }
    };
    uint4 ra[WG_NR], rb[WG_NR];
#pragma unroll
    for (int m = 0; m < WG_NR; m++) ra[m] = rb[m] = uint4{0u, 0u, 0u, 0u};
    load(p_lo, ra);
    if (p_lo + WG_PX < p_hi) load(p_lo + WG_PX, rb);
    for (long p0 = p_lo; p0 < p_hi; p0 += 2 * WG_PX) {
        tile(p0, ra);
        if (p0 + WG_PX < p_hi) tile(p0 + WG_PX, rb);
    }
    if (is_x) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            float *dst = partial + ((long)blockIdx.z * 9 + 3 * w + d) * Cout * Cin;
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < 2; b++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        dst[(long)(co0 + 16 * a + 4 * kq + i) * Cin + ci0 + 16 * b + r16] = acc[d][a][b][i];
        }
    } else if (do_b) {
        part_b[(long)blockIdx.z * Cout + co0 + lane] = bsum;
    }
}

// out[k] = sum_z partial[z][k] in z order; out2 likewise from partial2 (n2 entries)
__global__ void k_reduce_chunks(const float *__restrict__ partial, long n, int nz, float *__restrict__ out,
                                const float *__restrict__ partial2, long n2, float *__restrict__ out2)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n + n2) return;
    const bool first = k < n;
    const float *p = first ? partial + k : partial2 + (k - n);
    const long stride = first ? n : n2;
    float s = 0.0f;
#pragma unroll 16   // loads of 16 chunks in flight, the additions in z order
    for (int z = 0; z < nz; z++) s += p[(long)z * stride];
    (first ? out[k] : out2[k - n]) = s;
}

// Plain GEMM C[m][n] = sum_k A[m][k] B[n][k] (both K-contiguous, BF16; M, N
// multiples of 16, K of 32): one wave per 16 x 16 tile.  Exposes the MFMA
// fragment layout for testing.
__global__ __launch_bounds__(64) void k_gemm_bf16(const bf16_t *__restrict__ A, const bf16_t *__restrict__ B,
                                                  float *__restrict__ C, int M, int N, int K)
{
    const int lane = threadIdx.x, r16 = lane & 15, kq = lane >> 4;
    const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 32) {
        Frag a, b;
        a.raw = *(const uint4 *)(A + (long)(m0 + r16) * K + k0 + 8 * kq);
        b.raw = *(const uint4 *)(B + (long)(n0 + r16) * K + k0 + 8 * kq);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, b.v, acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) C[(long)(m0 + 4 * kq + i) * N + n0 + r16] = acc[i];
}

// ---------------------------------------------------------------------------
// element-wise and small kernels
// ---------------------------------------------------------------------------
// [9][Cout][Cin] FP32 -> BF16 copy, and the data-gradient weights
// Wf[8 - t][ci][co] = W[t][co][ci]
__global__ void k_prep_weights(const float *__restrict__ Wm, int Cout, int Cin, bf16_t *__restrict__ Wb,
                               bf16_t *__restrict__ Wf)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long n = 9L * Cout * Cin;
    if (k >= n) return;
    const int ci = (int)(k % Cin);
    const long r = k / Cin;
    const int co = (int)(r % Cout), t = (int)(r / Cout);
    bf16_t h = f2bf(Wm[k]);
    Wb[k] = h;
    if (Wf) Wf[((long)(8 - t) * Cin + ci) * Cout + co] = h;
}

// dz = bf16(dy * (y > 0))  (ReLU backward from the post-activation output)
__global__ void k_relu_bwd(const float *__restrict__ dy, const bf16_t *__restrict__ y, long n, bf16_t *__restrict__ dz)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) dz[k] = f2bf(bf2f(y[k]) > 0.0f ? dy[k] : 0.0f);
}

// 2x2 average pooling, NHWC
__global__ void k_pool2(const bf16_t *__restrict__ x, int N, int H, int W, int C, bf16_t *__restrict__ y)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int Ho = H / 2, Wo = W / 2;
    if (k >= (long)N * Ho * Wo * C) return;
    const int c = (int)(k % C);
    long r = k / C;
    const int xo = (int)(r % Wo);
    r /= Wo;
    const int yo = (int)(r % Ho), n = (int)(r / Ho);
    const long b = (((long)n * H + 2 * yo) * W + 2 * xo) * C + c;
    float s = ((bf2f(x[b]) + bf2f(x[b + C])) + bf2f(x[b + (long)W * C])) + bf2f(x[b + (long)W * C + C]);
    y[k] = f2bf(0.25f * s);
}
__global__ void k_pool2_bwd(const float *__restrict__ dy, int N, int H, int W, int C, float *__restrict__ dx, int acc)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)N * H * W * C) return;
    const int c = (int)(k % C);
    long r = k / C;
    const int x = (int)(r % W);
    r /= W;
    const int y = (int)(r % H), n = (int)(r / H);
    const float g = 0.25f * dy[(((long)n * (H / 2) + y / 2) * (W / 2) + x / 2) * C + c];
    dx[k] = acc ? dx[k] + g : g;
}
// 2x2 average pooling over 8-channel groups (C % 8 == 0, 16-byte aligned
// tensors): per channel the same sums as k_pool2
__global__ void k_pool2_v8(const bf16_t *__restrict__ x, int N, int H, int W, int C, bf16_t *__restrict__ y)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int Ho = H / 2, Wo = W / 2, C8 = C / 8;
    if (k >= (long)N * Ho * Wo * C8) return;
    const int c8 = (int)(k % C8);
    long r = k / C8;
    const int xo = (int)(r % Wo);
    r /= Wo;
    const int yo = (int)(r % Ho), n = (int)(r / Ho);
    const long b = (((long)n * H + 2 * yo) * W + 2 * xo) * C + 8 * c8;
    Bf8 q0, q1, q2, q3, o;
    q0.raw = *(const uint4 *)(x + b);
    q1.raw = *(const uint4 *)(x + b + C);
    q2.raw = *(const uint4 *)(x + b + (long)W * C);
    q3.raw = *(const uint4 *)(x + b + (long)W * C + C);
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float s = ((bf2f(q0.h[i]) + bf2f(q1.h[i])) + bf2f(q2.h[i])) + bf2f(q3.h[i]);
        o.h[i] = f2bf(0.25f * s);
    }
    *(uint4 *)(y + 8 * k) = o.raw;
}
// nearest x2 upsampling over 8-channel groups (C % 8 == 0, aligned)
__global__ void k_up2_v8(const bf16_t *__restrict__ x, int N, int H, int W, int C, bf16_t *__restrict__ y)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int C8 = C / 8;
    if (k >= (long)N * 4 * H * W * C8) return;
    const int c8 = (int)(k % C8);
    long r = k / C8;
    const int xo = (int)(r % (2 * W));
    r /= 2 * W;
    const int yo = (int)(r % (2 * H)), n = (int)(r / (2 * H));
    *(uint4 *)(y + 8 * k) = *(const uint4 *)(x + (((long)n * H + yo / 2) * W + xo / 2) * C + 8 * c8);
}
// nearest x2 upsampling, NHWC (input N x H x W)
__global__ void k_up2(const bf16_t *__restrict__ x, int N, int H, int W, int C, bf16_t *__restrict__ y)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)N * 4 * H * W * C) return;
    const int c = (int)(k % C);
    long r = k / C;
    const int xo = (int)(r % (2 * W));
    r /= 2 * W;
    const int yo = (int)(r % (2 * H)), n = (int)(r / (2 * H));
    y[k] = x[(((long)n * H + yo / 2) * W + xo / 2) * C + c];
}
// The backward passes that end at a ReLU's output: the gradient of 8 channels
// formed as the FP32 kernels form it, masked and rounded to BF16 at once
// (dz = bf16(y > 0 ? g : 0)); C % 8 == 0, tensors 16-byte aligned.  Bound by
// memory: the FP32 gradient is neither written nor read again.  Level 0 of a
// 16 x 256^2 training step: pooling 216 -> 52 us with its ReLU, the head's 157
// -> 23 us, upsampling onto level 1 62 -> 41 us.
__device__ __forceinline__ void relu_store(const float g[8], const bf16_t *y, bf16_t *dz)
{
    Bf8 a, o;
    a.raw = *(const uint4 *)y;
#pragma unroll
    for (int i = 0; i < 8; i++) o.h[i] = f2bf(bf2f(a.h[i]) > 0.0f ? g[i] : 0.0f);
    *(uint4 *)dz = o.raw;
}
__device__ __forceinline__ void load8(const float *p, float v[8])
{
    const float4 a = *(const float4 *)p, b = *(const float4 *)(p + 4);
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
// g + 0.25 dy (k_pool2_bwd accumulating into g)
__global__ void k_pool2_bwd_relu(const float *__restrict__ dy, const float *__restrict__ g, int N, int H, int W, int C,
                                 const bf16_t *__restrict__ y, bf16_t *__restrict__ dz)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int C8 = C / 8;
    if (k >= (long)N * H * W * C8) return;
    const int c8 = (int)(k % C8);
    long r = k / C8;
    const int px = (int)(r % W);
    r /= W;
    const int py = (int)(r % H), n = (int)(r / H);
    float d[8], a[8];
    load8(dy + (((long)n * (H / 2) + py / 2) * (W / 2) + px / 2) * C + 8 * c8, d);
    load8(g + 8 * k, a);
#pragma unroll
    for (int i = 0; i < 8; i++) a[i] = a[i] + 0.25f * d[i];
    relu_store(a, y + 8 * k, dz + 8 * k);
}
// k_up2_bwd
__global__ void k_up2_bwd_relu(const float *__restrict__ dy, int N, int H, int W, int C, const bf16_t *__restrict__ y,
                               bf16_t *__restrict__ dz)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int C8 = C / 8;
    if (k >= (long)N * H * W * C8) return;
    const int c8 = (int)(k % C8);
    long r = k / C8;
    const int px = (int)(r % W);
    r /= W;
    const int py = (int)(r % H), n = (int)(r / H);
    const long W2 = 2L * W, b = (((long)n * 2 * H + 2 * py) * W2 + 2 * px) * C + 8 * c8;
    float q0[8], q1[8], q2[8], q3[8];
    load8(dy + b, q0);
    load8(dy + b + C, q1);
    load8(dy + b + W2 * C, q2);
    load8(dy + b + W2 * C + C, q3);
#pragma unroll
    for (int i = 0; i < 8; i++) q0[i] = ((q0[i] + q1[i]) + q2[i]) + q3[i];
    relu_store(q0, y + 8 * k, dz + 8 * k);
}
// k_head_bwd_x; x is the head's input, the ReLU's output
template <int NO>
__global__ void k_head_bwd_relu(const float *__restrict__ dout, const bf16_t *__restrict__ x, long P, int C,
                                const float *__restrict__ Wh, bf16_t *__restrict__ dz)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int C8 = C / 8;
    if (k >= P * C8) return;
    const long p = k / C8;
    const int c = 8 * (int)(k - p * C8);
    float g[8];
#pragma unroll
    for (int o = 0; o < NO; o++) {
        const float d = dout[NO * p + o];
#pragma unroll
        for (int i = 0; i < 8; i++) g[i] = o ? g[i] + d * Wh[o * C + c + i] : d * Wh[c + i];
    }
    relu_store(g, x + 8 * k, dz + 8 * k);
}

__global__ void k_up2_bwd(const float *__restrict__ dy, int N, int H, int W, int C, float *__restrict__ dx)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)N * H * W * C) return;
    const int c = (int)(k % C);
    long r = k / C;
    const int x = (int)(r % W);
    r /= W;
    const int y = (int)(r % H), n = (int)(r / H);
    const long W2 = 2L * W;
    const long b = (((long)n * 2 * H + 2 * y) * W2 + 2 * x) * C + c;
    dx[k] = ((dy[b] + dy[b + C]) + dy[b + W2 * C]) + dy[b + W2 * C + C];
}

// bias gradient partials: part[z][c] = sum over pixel chunk z of dz[p][c]
__global__ void k_bias_grad(const bf16_t *__restrict__ dz, long P, int C, long chunk, float *__restrict__ part)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C) return;
    const long lo = (long)blockIdx.y * chunk, hi = lo + chunk < P ? lo + chunk : P;
    float s = 0.0f;
    for (long p = lo; p < hi; p++) s += bf2f(dz[p * C + c]);
    part[(long)blockIdx.y * C + c] = s;
}

// k_bias_grad for 16-byte aligned dz with C % 8 == 0: the same sums in the
// same pixel order.  The sum of a channel over a chunk is a serial chain of
// additions (so its rounding does not depend on the launch); one lane per
// channel that loads each value itself waits out a load latency per pixel.
// Here the workgroup stages SUM_PX pixels x 64 channels in LDS with 16-byte
// loads, the next tile's loads in flight while the first wave adds, so the
// chain runs at the rate of LDS reads and additions.  In a training step of
// 16 x 256^2 the 13 bias gradients took 10.1 ms and the head's weight gradient
// 1.2 ms; the step went from 20.0 to 8.6 ms with both staged.
constexpr int SUM_PX = 256;
__global__ __launch_bounds__(256) void k_bias_grad_v8(const bf16_t *__restrict__ dz, long P, int C, long chunk,
                                                      float *__restrict__ part)
{
    __shared__ bf16_t t[SUM_PX][64];
    const int c0 = blockIdx.x * 64, nc = C - c0 < 64 ? C - c0 : 64, n8 = nc / 8;
    const long lo = (long)blockIdx.y * chunk, hi = lo + chunk < P ? lo + chunk : P;
    const int g = threadIdx.x & 7, row = threadIdx.x >> 3;   // 8-channel group, pixel row of the staging pass
    uint4 r[SUM_PX / 32];
    auto load = [&](long p0) {
#pragma unroll
        for (int q = 0; q < SUM_PX / 32; q++) {
            const long p = p0 + row + 32 * q;
            r[q] = g < n8 && p < hi ? *(const uint4 *)(dz + p * C + c0 + 8 * g) : uint4{0u, 0u, 0u, 0u};
        }
    };
    float s = 0.0f;
    load(lo);
    for (long p0 = lo; p0 < hi; p0 += SUM_PX) {
        __syncthreads();   // the previous tile has been added
#pragma unroll
        for (int q = 0; q < SUM_PX / 32; q++)
            if (g < n8) *(uint4 *)&t[row + 32 * q][8 * g] = r[q];
        __syncthreads();
        if (p0 + SUM_PX < hi) load(p0 + SUM_PX);
        if ((int)threadIdx.x < nc) {
            const int n = hi - p0 < SUM_PX ? (int)(hi - p0) : SUM_PX;
#pragma unroll 16
            for (int k = 0; k < n; k++) s += bf2f(t[k][threadIdx.x]);
        }
    }
    if ((int)threadIdx.x < nc) part[(long)blockIdx.y * C + c0 + threadIdx.x] = s;
}

// 1x1 output head with NO <= 4 outputs:
// out[p][o] = b[o] + sum_c Wh[o][c] x[p][c]  (FP32)
__global__ void k_head(const bf16_t *__restrict__ x, long P, int C, int NO, const float *__restrict__ Wh,
                       const float *__restrict__ bh, float *__restrict__ out)
{
    long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int o = 0; o < NO; o++) s[o] = bh[o];
    for (int c = 0; c < C; c++) {
        float v = bf2f(x[p * C + c]);
        for (int o = 0; o < NO; o++) s[o] += Wh[o * C + c] * v;
    }
    for (int o = 0; o < NO; o++) out[NO * p + o] = s[o];
}
// k_head reading 8 channels per 16-byte access (C % 8 == 0, aligned): the
// same sums in the same order
template <int NO>
__global__ void k_head_v8(const bf16_t *__restrict__ x, long P, int C, const float *__restrict__ Wh,
                          const float *__restrict__ bh, float *__restrict__ out)
{
    long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    float s[NO];
#pragma unroll
    for (int o = 0; o < NO; o++) s[o] = bh[o];
#pragma unroll 4
    for (int c = 0; c < C; c += 8) {
        Bf8 q;
        q.raw = *(const uint4 *)(x + p * C + c);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float v = bf2f(q.h[i]);
#pragma unroll
            for (int o = 0; o < NO; o++) s[o] += Wh[o * C + c + i] * v;
        }
    }
#pragma unroll
    for (int o = 0; o < NO; o++) out[NO * p + o] = s[o];
}
// dx[p][c] = sum_o dout[p][o] Wh[o][c]
__global__ void k_head_bwd_x(const float *__restrict__ dout, long P, int C, int NO, const float *__restrict__ Wh,
                             float *__restrict__ dx)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= P * C) return;
    const long p = k / C;
    const int c = (int)(k % C);
    float s = dout[NO * p] * Wh[c];
    for (int o = 1; o < NO; o++) s += dout[NO * p + o] * Wh[o * C + c];
    dx[k] = s;
}
// partials over pixel chunks of dWh[o][c] = sum_p dout[p][o] x[p][c] and dbh[o] = sum_p dout[p][o]
__global__ void k_head_bwd_w(const float *__restrict__ dout, const bf16_t *__restrict__ x, long P, int C, int NO,
                             long chunk, float *__restrict__ part)
{
    const int k = threadIdx.x;   // 0 .. NO*C + NO - 1
    const int nk = NO * C + NO;
    if (k >= nk) return;
    const long lo = (long)blockIdx.x * chunk, hi = lo + chunk < P ? lo + chunk : P;
    float s = 0.0f;
    if (k < NO * C) {
        const int o = k / C, c = k % C;
        for (long p = lo; p < hi; p++) s += dout[NO * p + o] * bf2f(x[p * C + c]);
    } else {
        const int o = k - NO * C;
        for (long p = lo; p < hi; p++) s += dout[NO * p + o];
    }
    part[(long)blockIdx.x * nk + k] = s;
}

// k_head_bwd_w with both tensors staged in LDS (C % 16 == 0, C <= 64, x 16-byte
// aligned): the same sums in the same pixel order.  A lane's chain reads four
// pixels of its channel at once (ds_read_b64_tr_b16) and four of its output's
// gradient; the bias sums' lanes read a column of ones instead of x, so every
// lane runs the same chain.  16 x 256^2 pixels, 32 channels, 3 outputs: 1226
// us by k_head_bwd_w, 66 us by this.
constexpr int HB_NT = 320;   // threads: NO C + NO <= 260 chains
constexpr int HB_LD = 80;    // LDS pitch (bf16): up to 64 channels, 16 ones
template <int NO>
__global__ __launch_bounds__(HB_NT) void k_head_bwd_w_v8(const float *__restrict__ dout, const bf16_t *__restrict__ x,
                                                         long P, int C, long chunk, float *__restrict__ part)
{
    __shared__ bf16_t t[SUM_PX][HB_LD];
    __shared__ float d[4][SUM_PX];
    const int nk = NO * C + NO, n8 = C / 8, k = threadIdx.x, r16 = k & 15;
    const long lo = (long)blockIdx.x * chunk, hi = lo + chunk < P ? lo + chunk : P;
    constexpr int NX = (SUM_PX * 8 + HB_NT - 1) / HB_NT, ND = (SUM_PX * NO + HB_NT - 1) / HB_NT;
    uint4 r[NX];
    float rd[ND];
    auto load = [&](long p0) {
#pragma unroll
        for (int q = 0; q < NX; q++) {
            const int e = k + HB_NT * q, px = e / n8;
            r[q] = px < SUM_PX && p0 + px < hi ? *(const uint4 *)(x + (p0 + px) * C + 8 * (e - px * n8)) : uint4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int q = 0; q < ND; q++) {
            const int e = k + HB_NT * q;
            rd[q] = e < SUM_PX * NO && NO * p0 + e < NO * hi ? dout[NO * p0 + e] : 0.0f;
        }
    };
    for (int e = k; e < SUM_PX * 16; e += HB_NT) t[e >> 4][64 + (e & 15)] = 0x3f80;   // 1.0
    const bool prod = k < NO * C;
    const int o = prod ? k / C : (k < nk ? k - NO * C : 0), c16 = prod ? k % C - r16 : 64;
    const bf16_t *tc = &t[r16 >> 2][c16 + 4 * (r16 & 3)];
    float s = 0.0f;
    load(lo);
    for (long p0 = lo; p0 < hi; p0 += SUM_PX) {
        __syncthreads();   // the previous tile has been added
#pragma unroll
        for (int q = 0; q < NX; q++) {
            const int e = k + HB_NT * q, px = e / n8;
            if (px < SUM_PX) *(uint4 *)&t[px][8 * (e - px * n8)] = r[q];
        }
#pragma unroll
        for (int q = 0; q < ND; q++) {
            const int e = k + HB_NT * q;
            if (e < SUM_PX * NO) d[e % NO][e / NO] = rd[q];
        }
        __syncthreads();
        if (p0 + SUM_PX < hi) load(p0 + SUM_PX);
        if (k >= ((nk + 63) & ~63)) continue;   // a wave without a chain
        if (p0 + SUM_PX <= hi) {
#pragma unroll 8
            for (int q = 0; q < SUM_PX; q += 4) {
                const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(tc + q * HB_LD));
                const float4 g = *(const float4 *)&d[o][q];
                s += g.x * bf2f((bf16_t)v[0]);
                s += g.y * bf2f((bf16_t)v[1]);
                s += g.z * bf2f((bf16_t)v[2]);
                s += g.w * bf2f((bf16_t)v[3]);
            }
        } else {
            for (int q = 0; q < (int)(hi - p0); q++) s += d[o][q] * bf2f(t[q][c16 + r16]);
        }
    }
    if (k < nk) part[(long)blockIdx.x * nk + k] = s;
}

// masked mean-squared error: loss partials and d(loss)/d(pred) = 2 m (pred - target) / count
__global__ void k_mse(const float *__restrict__ pred, const float *__restrict__ target, const float *__restrict__ mask,
                      long n, float inv_count, float *__restrict__ grad, float *__restrict__ part)
{
    __shared__ float s[256];
    long k = (long)blockIdx.x * 256 + threadIdx.x;
    float e = 0.0f;
    if (k < n) {
        const float m = mask ? mask[k / 2] : 1.0f;
        const float d = (pred[k] - target[k]) * m;
        grad[k] = 2.0f * d * inv_count;
        e = d * d;
    }
    s[threadIdx.x] = e;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// Adam (FP32 master weights); bias corrections c1 = 1 - b1^t, c2 = 1 - b2^t
__device__ __forceinline__ float adam_update(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                                             float *__restrict__ v, long k, float lr, float b1, float b2, float eps,
                                             float c1, float c2, float wd)
{
    const float gk = g[k] + wd * w[k];
    const float mk = b1 * m[k] + (1.0f - b1) * gk;
    const float vk = b2 * v[k] + (1.0f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    return w[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
}
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, long n, float lr, float b1, float b2, float eps, float c1, float c2,
                       float wd)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) adam_update(w, g, m, v, k, lr, b1, b2, eps, c1, c2, wd);
}
// The step of many tensors with their BF16 copies (k_prep_weights) in one
// launch: the network's 28 tensors are a launch's overhead each (3.7 us of a step
// of 16 x 256^2, and its 13 weight copies 2.9 us; the step 2.03 -> 1.89 ms)
constexpr int ADAM_ITEMS = 32;
struct AdamArgs {
    GlideAdamItem it[ADAM_ITEMS];
    unsigned first[ADAM_ITEMS + 1];   // an item's first block
    int n;
};
__global__ __launch_bounds__(256) void k_adam_items(AdamArgs A, float lr, float b1, float b2, float eps, float c1, float c2,
                                                    float wd)
{
    int q = 0;
    while (q + 1 < A.n && blockIdx.x >= A.first[q + 1]) q++;
    const GlideAdamItem &I = A.it[q];
    const long k = (long)(blockIdx.x - A.first[q]) * 256 + threadIdx.x;
    if (k >= I.n) return;
    const float w = adam_update(I.w, I.g, I.m, I.v, k, lr, b1, b2, eps, c1, c2, wd);
    if (!I.wb) return;
    const int ci = (int)(k % I.cin);
    const long r = k / I.cin;
    const int co = (int)(r % I.cout), t = (int)(r / I.cout);
    const bf16_t h = f2bf(w);
    I.wb[k] = h;
    if (I.wflip) I.wflip[((long)(8 - t) * I.cin + ci) * I.cout + co] = h;
}

// ---------------------------------------------------------------------------
// solver <-> network
// ---------------------------------------------------------------------------
// Network input of one member, NHWC with 32 channels (7 used):
//   0: H / 1000, 1: tanh((bed + 0.917 H) / 200) (flotation margin: the way
//   the bed enters the momentum balance besides the surface), 2: 100 |grad s|,
//   3: log(beta) + 2, 4: B / 24 - 1, 5, 6: 100 ds/dx, 100 ds/dy (central
//   differences, one-sided at the edges); channels 7..31 are 0.  Every
//   channel is invariant to a shift of the domain, so a network trained on
//   small domains applies to large ones.
// s = max(bed, -0.917 H) + H (the reference's surface, glide/physics.py:223-229).
__device__ __forceinline__ double surf(const double *H, const double *bed, long k)
{
    return fmax(bed[k], -0.917 * H[k]) + H[k];
}
__global__ void k_features(const double *__restrict__ H, const double *__restrict__ bed, const double *__restrict__ beta,
                           const double *__restrict__ B, int ny, int nx, double dx, bf16_t *__restrict__ x)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long n = (long)ny * nx, k0 = k;
    k = k < n ? k : n - 1;
    const int i = (int)(k / nx), j = (int)(k % nx);
    const int jl = j > 0 ? j - 1 : j, jr = j < nx - 1 ? j + 1 : j;
    const int it = i > 0 ? i - 1 : i, ib = i < ny - 1 ? i + 1 : i;
    const double sx = (surf(H, bed, (long)i * nx + jr) - surf(H, bed, (long)i * nx + jl)) / ((jr - jl) * dx);
    const double sy = (surf(H, bed, (long)ib * nx + j) - surf(H, bed, (long)it * nx + j)) / ((ib - it) * dx);
    float f[7] = {(float)(H[k] / 1000.0), (float)tanh((bed[k] + 0.917 * H[k]) / 200.0),
                  (float)(100.0 * sqrt(sx * sx + sy * sy)), (float)(log(beta[k]) + 2.0), (float)(B[k] / 24.0 - 1.0),
                  (float)(100.0 * sx), (float)(100.0 * sy)};
    uint32_t h[8] = {};
#pragma unroll
    for (int c = 0; c < 7; c++) h[c] = f2bf(f[c]);
    const uint4 q = {h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6]};
    if ((uintptr_t)x & 15) {
        if (k0 < n)
            for (int c = 0; c < 32; c++) x[k * 32 + c] = (bf16_t)(c < 8 ? h[c & 7] : 0u);
        return;
    }
    // four consecutive lanes store one cell's 64 bytes
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int src = 16 * s + (lane >> 2);
        uint4 v = {(uint32_t)__shfl((int)q.x, src), (uint32_t)__shfl((int)q.y, src), (uint32_t)__shfl((int)q.z, src),
                   (uint32_t)__shfl((int)q.w, src)};
        if (lane & 3) v = uint4{0u, 0u, 0u, 0u};
        const long c = k0 - lane + src;
        if (c < n) *(uint4 *)(x + c * 32 + 8 * (lane & 3)) = v;
    }
}
// targets (FP32, 3 per cell): cell-centred (u_l + u_r)/2 and (v_t + v_b)/2
// times scale, and the thickness change (H - H_prev) times hscale
__global__ void k_targets(const double *__restrict__ u, const double *__restrict__ v, const double *__restrict__ H,
                          const double *__restrict__ H_prev, int ny, int nx, double scale, double hscale,
                          float *__restrict__ tgt)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= (long)ny * nx) return;
    const int i = (int)(k / nx), j = (int)(k % nx);
    tgt[3 * k] = (float)(0.5 * (u[(long)i * (nx + 1) + j] + u[(long)i * (nx + 1) + j + 1]) * scale);
    tgt[3 * k + 1] = (float)(0.5 * (v[(long)i * nx + j] + v[(long)(i + 1) * nx + j]) * scale);
    tgt[3 * k + 2] = (float)((H[k] - H_prev[k]) * hscale);
}
// the solver state from a prediction (3 per cell): faces from the cell-centred
// velocities / scale (interior faces average their two cells, boundary faces
// take their one cell); H = max(H_prev + dH / hscale, gamma)
__global__ void k_apply_prediction(const float *__restrict__ pred, int ny, int nx, double scale, double hscale,
                                   double *__restrict__ u, double *__restrict__ v, double *__restrict__ H,
                                   const double *__restrict__ H_prev, const double *__restrict__ gamma)
{
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long nu = (long)ny * (nx + 1), nv = (long)(ny + 1) * nx, nc = (long)ny * nx;
    if (k < nu) {
        const int i = (int)(k / (nx + 1)), j = (int)(k % (nx + 1));
        const int jl = j > 0 ? j - 1 : 0, jr = j < nx ? j : nx - 1;
        u[k] = 0.5 * ((double)pred[3 * ((long)i * nx + jl)] + (double)pred[3 * ((long)i * nx + jr)]) / scale;
    } else if (k < nu + nv) {
        const long kk = k - nu;
        const int i = (int)(kk / nx), j = (int)(kk % nx);
        const int it = i > 0 ? i - 1 : 0, ib = i < ny ? i : ny - 1;
        v[kk] = 0.5 * ((double)pred[3 * ((long)it * nx + j) + 1] + (double)pred[3 * ((long)ib * nx + j) + 1]) / scale;
    } else if (k < nu + nv + nc) {
        const long kk = k - nu - nv;
        H[kk] = fmax(H_prev[kk] + (double)pred[3 * kk + 2] / hscale, gamma[kk]);
    }
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
namespace {
inline unsigned nblk(long n, int bs = 256) { return (unsigned)((n + bs - 1) / bs); }
inline hipStream_t SS(void *s) { return (hipStream_t)s; }
bool bad_ch(int c) { return c < 0 || c % 32 != 0 || c > 4096; }
// 8-channel (16-byte) accesses apply: C % 8 == 0 and both tensors 16-byte aligned
bool vec8(int C, const void *a, const void *b) { return C % 8 == 0 && (((uintptr_t)a | (uintptr_t)b) & 15) == 0; }
// head weight-gradient partials, glide_unet_bias_chunks(P) x (NO C + NO)
void head_bwd_w(const float *dout, const bf16_t *x, long P, int C, int NO, float *partial, hipStream_t st)
{
    const int nk = NO * C + NO;
    const unsigned nz = (unsigned)((P + 4095) / 4096);
    if (vec8(C, x, x) && C % 16 == 0 && C <= 64) {
        auto go = [&](auto no) {
            hipLaunchKernelGGL(k_head_bwd_w_v8<decltype(no)::value>, dim3(nz), dim3(HB_NT), 0, st, dout, x, P, C, 4096L,
                               partial);
        };
        if (NO == 1) return go(std::integral_constant<int, 1>{});
        if (NO == 2) return go(std::integral_constant<int, 2>{});
        if (NO == 3) return go(std::integral_constant<int, 3>{});
        return go(std::integral_constant<int, 4>{});
    }
    hipLaunchKernelGGL(k_head_bwd_w, dim3(nz), dim3(((nk + 63) / 64) * 64), 0, st, dout, x, P, C, NO, 4096L, partial);
}
// Output channels per wave (16 * NJ) of the direct 3x3 convolution over P
// pixels: the
// widest of 64, 32 and 16 that still gives at least 2048 waves (two per
// SIMD), else 16.  Small levels are bound by each wave's serial K loop, so
// they take more, narrower waves; large ones keep the input fragments'
// reuse across output channels.  The sums are the same for every width.
int conv_nj(long P, int C)
{
    const long pw = (long)nblk(P) * 4;   // 64-pixel waves
    for (int nj = 4; nj > 1; nj /= 2)
        if (C % (16 * nj) == 0 && pw * (C / (16 * nj)) >= 2048) return nj;
    return 1;
}
void pool2(const bf16_t *x, int N, int H, int W, int C, bf16_t *y, hipStream_t st)
{
    const long n = (long)N * (H / 2) * (W / 2) * C;
    if (vec8(C, x, y))
        hipLaunchKernelGGL(k_pool2_v8, dim3(nblk(n / 8)), dim3(256), 0, st, x, N, H, W, C, y);
    else
        hipLaunchKernelGGL(k_pool2, dim3(nblk(n)), dim3(256), 0, st, x, N, H, W, C, y);
}
struct ConvArgs {
    const bf16_t *xa;
    int CA, up;   // up: xa is at half the resolution
    const bf16_t *xb;
    int CB, N, H, W;
    const bf16_t *Wt;
    int Cout;
    const float *bias;
    int relu;
    const bf16_t *ya;
    bf16_t *out, *pool;
    float *ga;
    int SA, acc_a;
    float *gb;
    int acc_b;
};

template <int NW, int NG, int NCH, int MODE>
void conv_launch(const ConvArgs &c, hipStream_t st)
{
    const int tx = (c.W + CV_W - 1) / CV_W, tiles = tx * ((c.H + 2 * NW - 1) / (2 * NW));
    hipLaunchKernelGGL((k_conv3x3<NW, NG, NCH, MODE>), dim3((unsigned)((long)tiles * c.N), c.Cout / (32 * NG)),
                       dim3(64 * NW * NG), 0, st, c.xa, c.CA, c.up, c.xb, c.H, c.W, tx, tiles, c.Wt, c.Cout, c.bias,
                       c.relu, c.ya, c.out, c.pool, c.ga, c.SA, c.acc_a, c.gb, c.acc_b);
}
// Row pairs per workgroup (tile rows / 2), and whether the staged kernel is the
// faster one at all.  Its time goes with the pixels of its tiles, inside the
// image or not; the direct kernel's with the pixels that there are (at 2.2 times
// the price in its narrowest form, 1.7 with 96 -> 96 channels), down to some 84000
// pixels by 32 output channels (56000 with 128 and more input channels), below
// which it waits out its loads.  A staged pixel costs, in pixels of the direct
// kernel, 0.28 where the weights are staged too, 0.45 in the taller tiles with
// three chunks of input channels and one workgroup for all output channels, else
// 0.56 (measured over 1 to 4000 images of 1 to 64 pixels a side and strips of 500,
// 32 to 192 channels: of the two kernels the faster one or within 10% of it, but for
// some shapes near the line, up to 1.5 times).  The cheapest height that still
// gives a workgroup per CU is taken, the taller one of two (fewer halo rows), and
// the direct kernel where it costs less than that and the tiles have no CU each.  96 -> 96 channels: 4000 images of 2 x 2 pixels 236 us
// staged, 27 direct; 1000 of 8 x 8 62 and 45; 500 of 20 x 20 97 and 151; 256 of 32 x
// 32 70 and 189.
template <int NG, int NCH, int MODE>
bool conv_staged(const ConvArgs &c, hipStream_t st)
{
    constexpr bool TALL = conv_lds(4, NCH) <= 64 * 1024 || conv_wl(4, NG, NCH), MID = conv_lds(2, NCH) <= 64 * 1024;
    const long groups = c.Cout / 32, pixels = (long)c.N * c.H * c.W;
    int nw = 1;
    long wgs = 0;
    double cost = 0.0;
    auto height = [&](int k, bool has) {
        const long w = (long)((c.W + CV_W - 1) / CV_W) * ((c.H + 2 * k - 1) / (2 * k)) * c.N * (groups / NG);
        const double each = conv_wl(k, NG, NCH) ? 0.28 : NCH == 3 && groups == NG && k > 1 ? 0.45 : 0.56;
        const double x = each * w * (2 * k * CV_W) * NG / groups;
        if (!has || (k > 1 && w < 256) || (wgs && x >= cost)) return;
        nw = k, wgs = w, cost = x;
    };
    height(4, TALL);
    height(2, MID);
    height(1, true);
    const double price = conv_nj(pixels, c.Cout) > 1 ? 1.0 : NCH == 3 && groups == 3 ? 1.7 : 2.2;
    if (wgs > 256 && cost > std::max(price * pixels, (NCH < 4 ? 84e3 : 56e3) / groups)) return false;
    if constexpr (TALL)
        if (nw == 4) return conv_launch<4, NG, NCH, MODE>(c, st), true;
    if constexpr (MID)
        if (nw == 2) return conv_launch<2, NG, NCH, MODE>(c, st), true;
    return conv_launch<1, NG, NCH, MODE>(c, st), true;
}
// The workgroup's waves share the staged input among up to 3 groups of 32 output channels.
template <int NCH, int MODE>
bool conv_groups(const ConvArgs &c, hipStream_t st)
{
    const int ng = c.Cout / 32;
    if (ng % 3 == 0) return conv_staged<3, NCH, MODE>(c, st);
    if (ng % 2 == 0) return conv_staged<2, NCH, MODE>(c, st);
    return conv_staged<1, NCH, MODE>(c, st);
}
template <int NJ, int MODE>
void conv_direct(const ConvArgs &c, hipStream_t st)
{
    auto k = k_conv3x3_direct<NJ, MODE, false>;
    if constexpr (MODE == 0)
        if (c.up) k = k_conv3x3_direct<NJ, MODE, true>;
    hipLaunchKernelGGL(k, dim3(nblk((long)c.N * c.H * c.W), c.Cout / (16 * NJ)), dim3(256), 0, st, c.xa, c.CA, c.xb, c.CB,
                       c.N, c.H, c.W, c.Wt, c.Cout, c.bias, c.relu, c.ya, c.out, c.ga, c.SA, c.acc_a, c.gb, c.acc_b);
}
// The channel counts of the network's layers have a staged instance.  It reads
// the bias and stores in 16-byte pieces, which the direct kernel does not: a
// tensor off that alignment takes the direct kernel, and so do images that leave
// most of a tile empty (conv_staged).
template <int MODE>
void conv(ConvArgs c, hipStream_t st)
{
    const uintptr_t al = (uintptr_t)c.bias | (uintptr_t)c.ya | (uintptr_t)c.out | (uintptr_t)c.pool | (uintptr_t)c.ga |
                         (uintptr_t)c.gb;
    auto staged = [&] {
        if (al & 15) return false;
        switch ((c.CA + c.CB) / 32) {
        case 1: return conv_groups<1, MODE>(c, st);
        case 2: return conv_groups<2, MODE>(c, st);
        case 3: return conv_groups<3, MODE>(c, st);
        case 4: return conv_groups<4, MODE>(c, st);
        case 6: return conv_groups<6, MODE>(c, st);
        }
        return false;
    };
    if (staged()) return;
    switch (conv_nj((long)c.N * c.H * c.W, c.Cout)) {
    case 4: conv_direct<4, MODE>(c, st); break;
    case 2: conv_direct<2, MODE>(c, st); break;
    default: conv_direct<1, MODE>(c, st);
    }
    if (c.pool) pool2(c.out, c.N, c.H, c.W, c.Cout, c.pool, st);
}
}  // namespace

extern "C" {

int glide_unet_conv3x3(const uint16_t *xa, int CA, const uint16_t *xb, int CB, int N, int H, int W,
                       const uint16_t *weights, int Cout, const float *bias, int relu, uint16_t *out, void *stream)
{
    if (!xa || !weights || !bias || !out || (CB > 0 && !xb)) return ufail(GLIDE_E_NULL, "conv3x3: NULL argument");
    if (bad_ch(CA) || CA == 0 || bad_ch(CB) || bad_ch(Cout) || Cout == 0 || N < 1 || H < 1 || W < 1)
        return ufail(GLIDE_E_SIZE, "conv3x3: channels must be positive multiples of 32, sizes positive");
    conv<0>(ConvArgs{xa, CA, 0, xb, CB, N, H, W, weights, Cout, bias, relu, nullptr, out, nullptr, nullptr, 0, 0, nullptr,
                     0}, SS(stream));
    return ucheck("conv3x3");
}

int glide_unet_conv3x3_up_pool(const uint16_t *xa, int CA, int up_a, const uint16_t *xb, int CB, int N, int H, int W,
                               const uint16_t *weights, int Cout, const float *bias, int relu, uint16_t *out,
                               uint16_t *pooled, void *stream)
{
    if (!xa || !weights || !bias || !out || (CB > 0 && !xb)) return ufail(GLIDE_E_NULL, "conv3x3: NULL argument");
    if (bad_ch(CA) || CA == 0 || bad_ch(CB) || bad_ch(Cout) || Cout == 0 || N < 1 || H < 1 || W < 1)
        return ufail(GLIDE_E_SIZE, "conv3x3: channels must be positive multiples of 32, sizes positive");
    if ((up_a || pooled) && (H % 2 || W % 2)) return ufail(GLIDE_E_SIZE, "conv3x3: even sizes required");
    conv<0>(ConvArgs{xa, CA, up_a != 0, xb, CB, N, H, W, weights, Cout, bias, relu, nullptr, out, pooled, nullptr, 0, 0,
                     nullptr, 0}, SS(stream));
    return ucheck("conv3x3");
}

int glide_unet_conv3x3_dgrad(const uint16_t *dz, int Cout, int N, int H, int W, const uint16_t *wflip, int CA,
                             float *ga, int acc_a, int CB, float *gb, int acc_b, void *stream)
{
    if (!dz || !wflip || !ga || (CB > 0 && !gb)) return ufail(GLIDE_E_NULL, "conv3x3_dgrad: NULL argument");
    if (bad_ch(Cout) || Cout == 0 || bad_ch(CA) || CA == 0 || bad_ch(CB) || N < 1 || H < 1 || W < 1)
        return ufail(GLIDE_E_SIZE, "conv3x3_dgrad: channels must be positive multiples of 32, sizes positive");
    // the transposed convolution: CA + CB output channels
    conv<1>(ConvArgs{dz, Cout, 0, nullptr, 0, N, H, W, wflip, CA + CB, nullptr, 0, nullptr, nullptr, nullptr, ga, CA, acc_a,
                     gb, acc_b},
            SS(stream));
    return ucheck("conv3x3_dgrad");
}

int glide_unet_conv3x3_dgrad_relu(const uint16_t *dz, int Cout, int N, int H, int W, const uint16_t *wflip, int Cin,
                                  const uint16_t *y, uint16_t *dzin, void *stream)
{
    if (!dz || !wflip || !y || !dzin) return ufail(GLIDE_E_NULL, "conv3x3_dgrad_relu: NULL argument");
    if (dz == dzin) return ufail(GLIDE_E_ARG, "conv3x3_dgrad_relu: dz and dzin must be distinct");
    if (bad_ch(Cout) || Cout == 0 || bad_ch(Cin) || Cin == 0 || N < 1 || H < 1 || W < 1)
        return ufail(GLIDE_E_SIZE, "conv3x3_dgrad_relu: channels must be positive multiples of 32, sizes positive");
    conv<2>(ConvArgs{dz, Cout, 0, nullptr, 0, N, H, W, wflip, Cin, nullptr, 0, y, dzin, nullptr, nullptr, 0, 0, nullptr, 0},
            SS(stream));
    return ucheck("conv3x3_dgrad_relu");
}

long glide_unet_wgrad_chunks(int N, int H, int W) { return ((long)N * H * W + 4095) / 4096; }

int glide_unet_conv3x3_wgrad_bias(const uint16_t *dz, int Cout, const uint16_t *xa, int CA, const uint16_t *xb, int CB,
                                  int N, int H, int W, float *partial, float *dw, float *db, void *stream)
{
    if (!dz || !xa || !partial || !dw || (CB > 0 && !xb)) return ufail(GLIDE_E_NULL, "conv3x3_wgrad: NULL argument");
    if (bad_ch(Cout) || Cout == 0 || bad_ch(CA) || CA == 0 || bad_ch(CB) || N < 1 || H < 1 || W < 1)
        return ufail(GLIDE_E_SIZE, "conv3x3_wgrad: channels must be positive multiples of 32, sizes positive");
    const long chunk = 4096;
    const long nz = glide_unet_wgrad_chunks(N, H, W);
    const int Cin = CA + CB;
    const long n = 9L * Cout * Cin, n2 = db ? Cout : 0;
    float *part_b = db ? partial + nz * n : nullptr;
    hipLaunchKernelGGL(k_conv3x3_wgrad, dim3(Cin / 32, Cout / 32, (unsigned)nz), dim3(256), 0, SS(stream), dz, Cout, xa,
                       CA, xb, CB, N, H, W, chunk, partial, part_b);
    hipLaunchKernelGGL(k_reduce_chunks, dim3(nblk(n + n2)), dim3(256), 0, SS(stream), partial, n, (int)nz, dw, part_b, n2,
                       db);
    return ucheck("conv3x3_wgrad");
}

int glide_unet_conv3x3_wgrad(const uint16_t *dz, int Cout, const uint16_t *xa, int CA, const uint16_t *xb, int CB,
                             int N, int H, int W, float *partial, float *dw, void *stream)
{
    return glide_unet_conv3x3_wgrad_bias(dz, Cout, xa, CA, xb, CB, N, H, W, partial, dw, nullptr, stream);
}

int glide_unet_gemm_bf16(const uint16_t *A, const uint16_t *B, float *C, int M, int N, int K, void *stream)
{
    if (!A || !B || !C) return ufail(GLIDE_E_NULL, "gemm: NULL argument");
    if (M < 16 || N < 16 || K < 32 || M % 16 || N % 16 || K % 32)
        return ufail(GLIDE_E_SIZE, "gemm: M, N multiples of 16 and K a multiple of 32");
    hipLaunchKernelGGL(k_gemm_bf16, dim3(N / 16, M / 16), dim3(64), 0, SS(stream), A, B, C, M, N, K);
    return ucheck("gemm");
}

int glide_unet_prep_weights(const float *wm, int Cout, int Cin, uint16_t *wb, uint16_t *wflip, void *stream)
{
    if (!wm || !wb) return ufail(GLIDE_E_NULL, "prep_weights: NULL argument");
    if (Cout < 1 || Cin < 1) return ufail(GLIDE_E_SIZE, "prep_weights: bad shape");
    const long n = 9L * Cout * Cin;
    hipLaunchKernelGGL(k_prep_weights, dim3(nblk(n)), dim3(256), 0, SS(stream), wm, Cout, Cin, wb, wflip);
    return ucheck("prep_weights");
}

int glide_unet_relu_bwd(const float *dy, const uint16_t *y, long n, uint16_t *dz, void *stream)
{
    if (!dy || !y || !dz) return ufail(GLIDE_E_NULL, "relu_bwd: NULL argument");
    if (n < 0) return ufail(GLIDE_E_SIZE, "relu_bwd: negative size");
    if (n) hipLaunchKernelGGL(k_relu_bwd, dim3(nblk(n)), dim3(256), 0, SS(stream), dy, y, n, dz);
    return ucheck("relu_bwd");
}

int glide_unet_pool2(const uint16_t *x, int N, int H, int W, int C, uint16_t *y, void *stream)
{
    if (!x || !y) return ufail(GLIDE_E_NULL, "pool2: NULL argument");
    if (N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || C < 1) return ufail(GLIDE_E_SIZE, "pool2: even sizes required");
    pool2(x, N, H, W, C, y, SS(stream));
    return ucheck("pool2");
}

int glide_unet_pool2_bwd(const float *dy, int N, int H, int W, int C, float *dx, int accumulate, void *stream)
{
    if (!dy || !dx) return ufail(GLIDE_E_NULL, "pool2_bwd: NULL argument");
    if (N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || C < 1) return ufail(GLIDE_E_SIZE, "pool2_bwd: even sizes required");
    const long n = (long)N * H * W * C;
    hipLaunchKernelGGL(k_pool2_bwd, dim3(nblk(n)), dim3(256), 0, SS(stream), dy, N, H, W, C, dx, accumulate);
    return ucheck("pool2_bwd");
}

int glide_unet_up2(const uint16_t *x, int N, int H, int W, int C, uint16_t *y, void *stream)
{
    if (!x || !y) return ufail(GLIDE_E_NULL, "up2: NULL argument");
    if (N < 1 || H < 1 || W < 1 || C < 1) return ufail(GLIDE_E_SIZE, "up2: bad size");
    const long n = (long)N * 4 * H * W * C;
    if (vec8(C, x, y))
        hipLaunchKernelGGL(k_up2_v8, dim3(nblk(n / 8)), dim3(256), 0, SS(stream), x, N, H, W, C, y);
    else
        hipLaunchKernelGGL(k_up2, dim3(nblk(n)), dim3(256), 0, SS(stream), x, N, H, W, C, y);
    return ucheck("up2");
}

int glide_unet_up2_bwd(const float *dy, int N, int H, int W, int C, float *dx, void *stream)
{
    if (!dy || !dx) return ufail(GLIDE_E_NULL, "up2_bwd: NULL argument");
    if (N < 1 || H < 1 || W < 1 || C < 1) return ufail(GLIDE_E_SIZE, "up2_bwd: bad size");
    const long n = (long)N * H * W * C;
    hipLaunchKernelGGL(k_up2_bwd, dim3(nblk(n)), dim3(256), 0, SS(stream), dy, N, H, W, C, dx);
    return ucheck("up2_bwd");
}

long glide_unet_bias_chunks(long P) { return (P + 4095) / 4096; }

int glide_unet_bias_grad(const uint16_t *dz, long P, int C, float *partial, float *db, void *stream)
{
    if (!dz || !partial || !db) return ufail(GLIDE_E_NULL, "bias_grad: NULL argument");
    if (P < 1 || C < 1) return ufail(GLIDE_E_SIZE, "bias_grad: bad size");
    const long nz = glide_unet_bias_chunks(P);
    if (vec8(C, dz, dz))
        hipLaunchKernelGGL(k_bias_grad_v8, dim3((C + 63) / 64, (unsigned)nz), dim3(256), 0, SS(stream), dz, P, C,
                           4096L, partial);
    else
        hipLaunchKernelGGL(k_bias_grad, dim3((C + 63) / 64, (unsigned)nz), dim3(64), 0, SS(stream), dz, P, C, 4096L,
                           partial);
    hipLaunchKernelGGL(k_reduce_chunks, dim3(nblk(C)), dim3(256), 0, SS(stream), partial, (long)C, (int)nz, db,
                       (const float *)nullptr, 0L, (float *)nullptr);
    return ucheck("bias_grad");
}

int glide_unet_head(const uint16_t *x, long P, int C, int NO, const float *wh, const float *bh, float *out,
                    void *stream)
{
    if (!x || !wh || !bh || !out) return ufail(GLIDE_E_NULL, "head: NULL argument");
    if (P < 1 || C < 1 || NO < 1 || NO > 4) return ufail(GLIDE_E_SIZE, "head: bad size (1 <= outputs <= 4)");
    const dim3 grid(nblk(P)), block(256);
    hipStream_t st = SS(stream);
    if (!vec8(C, x, x))
        hipLaunchKernelGGL(k_head, grid, block, 0, st, x, P, C, NO, wh, bh, out);
    else if (NO == 1)
        hipLaunchKernelGGL(k_head_v8<1>, grid, block, 0, st, x, P, C, wh, bh, out);
    else if (NO == 2)
        hipLaunchKernelGGL(k_head_v8<2>, grid, block, 0, st, x, P, C, wh, bh, out);
    else if (NO == 3)
        hipLaunchKernelGGL(k_head_v8<3>, grid, block, 0, st, x, P, C, wh, bh, out);
    else
        hipLaunchKernelGGL(k_head_v8<4>, grid, block, 0, st, x, P, C, wh, bh, out);
    return ucheck("head");
}

int glide_unet_head_bwd(const float *dout, const uint16_t *x, long P, int C, int NO, const float *wh, float *dx,
                        float *partial, float *dwh_dbh, void *stream)
{
    if (!dout || !x || !wh || !dx || !partial || !dwh_dbh) return ufail(GLIDE_E_NULL, "head_bwd: NULL argument");
    const int nk = NO * C + NO;
    if (P < 1 || C < 1 || NO < 1 || NO > 4 || nk > 1024) return ufail(GLIDE_E_SIZE, "head_bwd: bad size");
    hipLaunchKernelGGL(k_head_bwd_x, dim3(nblk(P * C)), dim3(256), 0, SS(stream), dout, P, C, NO, wh, dx);
    const long nz = glide_unet_bias_chunks(P);
    head_bwd_w(dout, x, P, C, NO, partial, SS(stream));
    hipLaunchKernelGGL(k_reduce_chunks, dim3(nblk(nk)), dim3(256), 0, SS(stream), partial, (long)nk, (int)nz, dwh_dbh,
                       (const float *)nullptr, 0L, (float *)nullptr);
    return ucheck("head_bwd");
}

int glide_unet_head_bwd_relu(const float *dout, const uint16_t *x, long P, int C, int NO, const float *wh, uint16_t *dz,
                             float *partial, float *dwh_dbh, void *stream)
{
    if (!dout || !x || !wh || !dz || !partial || !dwh_dbh) return ufail(GLIDE_E_NULL, "head_bwd_relu: NULL argument");
    const int nk = NO * C + NO;
    if (P < 1 || C < 1 || C % 8 || NO < 1 || NO > 4 || nk > 1024) return ufail(GLIDE_E_SIZE, "head_bwd_relu: bad size");
    if (!vec8(C, x, dz)) return ufail(GLIDE_E_ARG, "head_bwd_relu: x and dz must be 16-byte aligned");
    const dim3 grid(nblk(P * (C / 8)));
    hipStream_t st = SS(stream);
    if (NO == 1) hipLaunchKernelGGL(k_head_bwd_relu<1>, grid, dim3(256), 0, st, dout, x, P, C, wh, dz);
    if (NO == 2) hipLaunchKernelGGL(k_head_bwd_relu<2>, grid, dim3(256), 0, st, dout, x, P, C, wh, dz);
    if (NO == 3) hipLaunchKernelGGL(k_head_bwd_relu<3>, grid, dim3(256), 0, st, dout, x, P, C, wh, dz);
    if (NO == 4) hipLaunchKernelGGL(k_head_bwd_relu<4>, grid, dim3(256), 0, st, dout, x, P, C, wh, dz);
    head_bwd_w(dout, x, P, C, NO, partial, st);
    hipLaunchKernelGGL(k_reduce_chunks, dim3(nblk(nk)), dim3(256), 0, st, partial, (long)nk,
                       (int)glide_unet_bias_chunks(P), dwh_dbh, (const float *)nullptr, 0L, (float *)nullptr);
    return ucheck("head_bwd_relu");
}

int glide_unet_pool2_bwd_relu(const float *dy, const float *g, int N, int H, int W, int C, const uint16_t *y,
                              uint16_t *dz, void *stream)
{
    if (!dy || !g || !y || !dz) return ufail(GLIDE_E_NULL, "pool2_bwd_relu: NULL argument");
    if (N < 1 || H < 2 || W < 2 || H % 2 || W % 2 || C < 8 || C % 8)
        return ufail(GLIDE_E_SIZE, "pool2_bwd_relu: even sizes and channels in multiples of 8 required");
    if (!vec8(C, dy, g) || !vec8(C, y, dz)) return ufail(GLIDE_E_ARG, "pool2_bwd_relu: tensors must be 16-byte aligned");
    hipLaunchKernelGGL(k_pool2_bwd_relu, dim3(nblk((long)N * H * W * (C / 8))), dim3(256), 0, SS(stream), dy, g, N, H, W,
                       C, y, dz);
    return ucheck("pool2_bwd_relu");
}

int glide_unet_up2_bwd_relu(const float *dy, int N, int H, int W, int C, const uint16_t *y, uint16_t *dz, void *stream)
{
    if (!dy || !y || !dz) return ufail(GLIDE_E_NULL, "up2_bwd_relu: NULL argument");
    if (N < 1 || H < 1 || W < 1 || C < 8 || C % 8)
        return ufail(GLIDE_E_SIZE, "up2_bwd_relu: positive sizes and channels in multiples of 8 required");
    if (!vec8(C, dy, y) || !vec8(C, dz, dz)) return ufail(GLIDE_E_ARG, "up2_bwd_relu: tensors must be 16-byte aligned");
    hipLaunchKernelGGL(k_up2_bwd_relu, dim3(nblk((long)N * H * W * (C / 8))), dim3(256), 0, SS(stream), dy, N, H, W, C, y,
                       dz);
    return ucheck("up2_bwd_relu");
}

long glide_unet_mse_blocks(long n) { return (n + 255) / 256; }

int glide_unet_mse(const float *pred, const float *target, const float *mask, long n, float inv_count, float *grad,
                   float *partial, void *stream)
{
    if (!pred || !target || !grad || !partial) return ufail(GLIDE_E_NULL, "mse: NULL argument");
    if (n < 1) return ufail(GLIDE_E_SIZE, "mse: empty");
    hipLaunchKernelGGL(k_mse, dim3((unsigned)glide_unet_mse_blocks(n)), dim3(256), 0, SS(stream), pred, target, mask, n,
                       inv_count, grad, partial);
    return ucheck("mse");
}

int glide_unet_adam(float *w, const float *g, float *m, float *v, long n, float lr, float b1, float b2, float eps,
                    int step, float weight_decay, void *stream)
{
    if (!w || !g || !m || !v) return ufail(GLIDE_E_NULL, "adam: NULL argument");
    if (n < 1 || step < 1) return ufail(GLIDE_E_SIZE, "adam: bad size or step");
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(nblk(n)), dim3(256), 0, SS(stream), w, g, m, v, n, lr, b1, b2, eps, c1, c2,
                       weight_decay);
    return ucheck("adam");
}

int glide_unet_adam_items(const GlideAdamItem *items, int n_items, float lr, float b1, float b2, float eps, int step,
                          float weight_decay, void *stream)
{
    if (!items) return ufail(GLIDE_E_NULL, "adam: NULL argument");
    if (n_items < 0 || step < 1) return ufail(GLIDE_E_SIZE, "adam: bad count or step");
    for (int q = 0; q < n_items; q++) {
        const GlideAdamItem &I = items[q];
        if (!I.w || !I.g || !I.m || !I.v) return ufail(GLIDE_E_NULL, "adam: NULL tensor");
        if (I.n < 1 || I.n > (1L << 32) || (I.wb && (I.cout < 1 || I.cin < 1 || I.n != 9L * I.cout * I.cin)))
            return ufail(GLIDE_E_SIZE, "adam: bad tensor size");
    }
    const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
    for (int q0 = 0; q0 < n_items; q0 += ADAM_ITEMS) {
        AdamArgs A;
        A.n = n_items - q0 < ADAM_ITEMS ? n_items - q0 : ADAM_ITEMS;
        unsigned blocks = 0;
        for (int q = 0; q < A.n; q++) {
            A.it[q] = items[q0 + q];
            A.first[q] = blocks;
            blocks += nblk(A.it[q].n);
        }
        A.first[A.n] = blocks;
        hipLaunchKernelGGL(k_adam_items, dim3(blocks), dim3(256), 0, SS(stream), A, lr, b1, b2, eps, c1, c2, weight_decay);
    }
    return ucheck("adam");
}

int glide_unet_features(const double *H, const double *bed, const double *beta, const double *B, int ny, int nx,
                        double dx, uint16_t *x, void *stream)
{
    if (!H || !bed || !beta || !B || !x) return ufail(GLIDE_E_NULL, "features: NULL argument");
    if (ny < 2 || nx < 2 || !(dx > 0.0)) return ufail(GLIDE_E_SIZE, "features: bad grid");
    const long n = (long)ny * nx;
    hipLaunchKernelGGL(k_features, dim3(nblk(n)), dim3(256), 0, SS(stream), H, bed, beta, B, ny, nx, dx, x);
    return ucheck("features");
}

int glide_unet_targets(const double *u, const double *v, const double *H, const double *H_prev, int ny, int nx,
                       double scale, double hscale, float *tgt, void *stream)
{
    if (!u || !v || !H || !H_prev || !tgt) return ufail(GLIDE_E_NULL, "targets: NULL argument");
    if (ny < 1 || nx < 1) return ufail(GLIDE_E_SIZE, "targets: bad grid");
    hipLaunchKernelGGL(k_targets, dim3(nblk((long)ny * nx)), dim3(256), 0, SS(stream), u, v, H, H_prev, ny, nx, scale,
                       hscale, tgt);
    return ucheck("targets");
}

int glide_unet_apply_prediction(const float *pred, int ny, int nx, double scale, double hscale, double *u, double *v,
                                double *H, const double *H_prev, const double *gamma, void *stream)
{
    if (!pred || !u || !v || !H || !H_prev || !gamma) return ufail(GLIDE_E_NULL, "apply_prediction: NULL argument");
    if (ny < 1 || nx < 1 || !(scale > 0.0) || !(hscale > 0.0))
        return ufail(GLIDE_E_SIZE, "apply_prediction: bad grid or scale");
    const long n = (long)ny * (nx + 1) + (long)(ny + 1) * nx + (long)ny * nx;
    hipLaunchKernelGGL(k_apply_prediction, dim3(nblk(n)), dim3(256), 0, SS(stream), pred, ny, nx, scale, hscale, u, v,
                       H, H_prev, gamma);
    return ucheck("apply_prediction");
}

}  // extern "C"
