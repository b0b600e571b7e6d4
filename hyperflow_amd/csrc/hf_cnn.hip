// hf_cnn.hip -- gfx950 kernels of the learned coarse-grid correction:
// BF16 MFMA 3x3 convolutions (forward, data gradient, weight gradient) with
// FP32 accumulation, input packing with a shock sensor, the loss, gradient
// reduction, Adam, weight packing, and the state transfers between the
// solver and the network.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hf_cnn.h"

namespace hfn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// FP32 -> BF16, round to nearest even (NaN -> quiet NaN).
__device__ __forceinline__ uint16_t f2bf(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0u;
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint32_t h) { return __uint_as_float(h << 16); }

__device__ __forceinline__ bf16x8 load8(const uint16_t* p)
{
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ bf16x8 zero8()
{
    const uint4 v = make_uint4(0u, 0u, 0u, 0u);
    return __builtin_bit_cast(bf16x8, v);
}

// Two FP32 values as packed BF16, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// A workgroup barrier for data in LDS: waits for this wave's LDS operations
// only.  (__syncthreads also waits for global loads and stores, here those of
// rows that are not needed before the next step.)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Output channels 0..3 of pixel (x, y): stored, or applied to the solver state
// (u, and its shock flag, requested earlier) with the fallbacks.
template <int MODE>
__device__ __forceinline__ void output(const NetArgs& a, int x, int y, const f32x4& acc, const float (&bias)[4],
                                       const float (&u)[4], uint32_t shock, uint32_t& nfb)
{
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = acc[r] + bias[r];
    if (MODE == NET_OUT_PLANES) {
        const int64_t np = (int64_t)a.nx * a.ny;
#pragma unroll
        for (int r = 0; r < 4; r++) (a.outf + r * np + (int64_t)y * a.nx)[(uint32_t)x] = v[r];
        return;
    }
    float n[4];
#pragma unroll
    for (int r = 0; r < 4; r++) n[r] = u[r] + a.scale[r] * v[r];
    const float p = (a.gamma - 1.0f) * (n[3] - 0.5f * (n[1] * n[1] + n[2] * n[2]) / n[0]);
    bool inrange = true;
    if (a.max_output > 0.0f)
#pragma unroll
        for (int r = 0; r < 4; r++) inrange = inrange && fabsf(v[r]) <= a.max_output;
    const bool ok = n[0] > 0.0f && p > 0.0f && !shock && inrange && isfinite(p) && isfinite(n[1]) && isfinite(n[2]) &&
                    isfinite(n[3]);
    if (ok) {
#pragma unroll
        for (int r = 0; r < 4; r++) (a.U + r * a.plane + (int64_t)y * a.pitch)[(uint32_t)x] = n[r];
    } else {
        nfb++;
    }
}

// ----------------------------------------------------------------- network --
// The whole forward pass of an 80-column strip in one workgroup of 8 waves,
// streaming down its rows: at step s, layer k works on row yc - 4 + s -
// 2 (k - 1), one row of every layer side by side, and a barrier ends the step.
// A hidden row goes to LDS (two slots per layer; four after layer 4), from
// where the next layer reads it one step later; nothing but the packed input
// and the output touches memory (STORE: also each activation's own pixels, for
// the backward pass).
//  * Frame: 96 columns from 8 left of the strip, six 16-pixel segments; each
//    layer's outermost columns are junk that the next one keeps away from (4
//    columns of halo per side, 8 kept for alignment).
//  * Waves 0-5: layers 2-4, two waves each, three segments per wave.  Layer k's
//    18 weight operands stay in registers, and so does the 3-row window of its
//    input (a ring of rows named at compile time: three LDS reads per segment
//    and row).  Waves 6-7: layer 1 (input rows requested three steps ahead and
//    kept in LDS) and layer 5 (window read from LDS), in one piece of code.
//  * An MFMA is 16x16x32: A = weights (rows = output channels), B = 32 input
//    values of 16 pixels.  Lane (g = lane/16, j = lane%16) feeds pixel j and K
//    chunk g and receives channels 16 mt + 4g + r.  For 32 input channels an
//    MFMA is one tap; for 8, K chunk 4s + g is tap 4s + g.  Pixels outside the
//    image are stored as zeros ("same" padding of every layer).
// Bound by the step's chain (LDS reads, 54 MFMAs per wave with two waves per
// SIMD, the epilogue, the barrier: about 3 000 cycles of which the MFMAs fill
// 1 728), H + 12 steps.  As five launches, each layer wrote and read 64 bytes a
// pixel (27 us of memory time per layer, 40 taken).  us for planes at 1024^2,
// corrected state at 1024^2, stored activations at 256^2:
//   five launches                                          169   188   27
//   one, rows as 64 bytes a pixel, __syncthreads()         128   181
//   barrier that waits for LDS only                        120   172   26
//   a plane per K chunk (NetRow)                           111   171   24.2
//   layer 1's input through LDS, state requested ahead     107   142   23.4
//   waves 6-7 first (without layer 5 a step would be a quarter shorter)
//                                                           97   132   22.6
// Layer 5's window in registers: 100, but 161 (spills); without the conditions
// that leave out a strip's unused steps the third column is 30.
constexpr int NET_OUT = 80, NET_SEGS = 6;
// A hidden row in LDS: a plane per K chunk (8 channels, 16 bytes a pixel), its
// 98 pixels padded to a multiple of the 256 bytes of a pass over the banks.
// Reads (16 lanes with consecutive pixels of one plane) and writes (8 bytes)
// then touch every bank once; with a pixel's 64 bytes together 74 % of the LDS
// cycles were conflicts (21 % now).
constexpr int NET_PX = 112;
typedef uint16_t NetRow[4][NET_PX][8];

template <int MODE, bool STORE>
__global__ __launch_bounds__(512, 2) void k_net(const NetArgs a)
{
    __shared__ __attribute__((aligned(256))) NetRow buf[10];
    __shared__ __attribute__((aligned(256))) uint16_t input[2][4][50][8];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, j = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nstrip = (a.nx + NET_OUT - 1) / NET_OUT;
    const int X0 = (int)(blockIdx.x % nstrip) * NET_OUT - 8;
    const int yc = (int)(blockIdx.x / nstrip) * a.rows, ye = min(a.ny, yc + a.rows);
    const int W2 = a.nx + 2;
    const int steps = (ye - yc + 12 + 2) / 3 * 3;   // the waves' loops advance by three

    // A 16-pixel segment of a hidden row: bias, ReLU, BF16, zeros outside the
    // image, into an LDS row and (STORE) the stored activation.
    auto finish = [&](int k, int row, int f0, const f32x4 (&acc)[2], const float (&bias)[2][4], NetRow& dst) {
        const int f = f0 + j, x = X0 + f;
        const bool in = x >= 0 && x < a.nx && row >= 0 && row < a.ny;
#pragma unroll
        for (int mt = 0; mt < 2; mt++) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = fmaxf(acc[mt][r] + bias[mt][r], 0.0f);
            uint2 pk;
            pk.x = in ? pk_bf16(v[0], v[1]) : 0u;
            pk.y = in ? pk_bf16(v[2], v[3]) : 0u;
            *reinterpret_cast<uint2*>(&dst[2 * mt + (g >> 1)][f + 1][4 * (g & 1)]) = pk;
            if (STORE && in && f >= 8 && f < 8 + NET_OUT && row >= yc && row < ye)
                *reinterpret_cast<uint2*>(a.act[k - 1] + ((size_t)(row + 1) * W2 + x + 1) * 32 + 16 * mt + 4 * g) = pk;
        }
    };
    auto load_bias = [&](int k, float (&bias)[2][4]) {
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++) bias[mt][r] = a.bias[k - 1][16 * mt + 4 * g + r];
    };
    uint32_t nfb = 0;

    if (wave < 6) {   // layers 2-4
        const int k = 2 + (wave >> 1), f0 = (wave & 1) * 48;
        bf16x8 wA[2][9];
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int t = 0; t < 9; t++) wA[mt][t] = load8(a.w[k - 1] + ((size_t)(mt * 9 + t) * 64 + lane) * 8);
        float bias[2][4];
        load_bias(k, bias);
        bf16x8 ring[3][3][3];   // [row][segment][column shift]
        for (int s0 = 0; s0 < steps; s0 += 3) {
#pragma unroll
            for (int ph = 0; ph < 3; ph++) {
                const int s = s0 + ph;
                const NetRow& src = buf[2 * (k - 2) + ((s + 1) & 1)];   // written last step
#pragma unroll
                for (int q = 0; q < 3; q++)
#pragma unroll
                    for (int d = 0; d < 3; d++) ring[ph][q][d] = load8(src[g][f0 + 16 * q + j + d]);
                const int row = yc - 4 + s - 2 * (k - 1);
                if (row >= yc - (5 - k) && row < ye + (5 - k)) {
                    NetRow& dst = buf[k < 4 ? 2 * (k - 1) + (s & 1) : 6 + (s & 3)];
#pragma unroll
                    for (int q = 0; q < 3; q++) {   // a segment's epilogue runs beside the next one's MFMAs
                        f32x4 acc[2] = {f32x4{0.0f, 0.0f, 0.0f, 0.0f}, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
                        for (int t = 0; t < 9; t++)
#pragma unroll
                            for (int mt = 0; mt < 2; mt++)
                                acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                    wA[mt][t], ring[(ph + 1 + t / 3) % 3][q][t % 3], acc[mt], 0, 0, 0);
                        finish(k, row, f0 + 16 * q, acc, bias, dst);
                    }
                }
                lds_barrier();
            }
        }
    } else {          // layers 1 and 5
        __builtin_amdgcn_s_setprio(2);   // the longest chain of a step: first choice beside waves 2 and 3
        const int h = wave - 6, f0 = h * 48;
        bf16x8 w1[2][3], w5[9];
#pragma unroll
        for (int mt = 0; mt < 2; mt++)
#pragma unroll
            for (int t = 0; t < 3; t++) w1[mt][t] = load8(a.w[0] + ((size_t)(mt * 3 + t) * 64 + lane) * 8);
#pragma unroll
        for (int t = 0; t < 9; t++) w5[t] = load8(a.w[4] + ((size_t)t * 64 + lane) * 8);
        float bias[2][4], b5[4];
        load_bias(1, bias);
#pragma unroll
        for (int r = 0; r < 4; r++) b5[r] = g == 0 ? a.bias[4][r] : 0.0f;
        // Layer 1's input: each wave keeps the 50 pixels of its segments, four
        // rows of them, in its own part of LDS; a row is requested three steps
        // before it is put there and read.  Pixels outside the padded image
        // (which only junk columns and rows reach) read its nearest ones.
        uint16_t (*const img)[50][8] = input[h];
        const uint32_t xoff = (uint32_t)min(max(X0 + f0 + min(lane, 49), 0), a.nx + 1) * 8u;
        auto fetch = [&](int row) {
            return load8(a.x + (size_t)min(max(row, 0), a.ny + 1) * ((size_t)W2 * 8) + xoff);
        };
        auto keep = [&](int row, const bf16x8& v) {
            if (lane < 50) *reinterpret_cast<bf16x8*>(img[row & 3][lane]) = v;
        };
        int tap[3];
#pragma unroll
        for (int t = 0; t < 3; t++) tap[t] = min(4 * t + g, 8);
        // the state under layer 5's output pixels (lanes g = 0)
        auto fetch_state = [&](int row, float (&u)[3][4], uint32_t (&shock)[3]) {
            if (MODE != NET_APPLY) return;
            const int y = min(max(row, yc), ye - 1);
#pragma unroll
            for (int q = 0; q < 3; q++) {
                const uint32_t x = (uint32_t)min(X0 + 8 + 16 * (3 * h + q) + j, a.nx - 1);
#pragma unroll
                for (int r = 0; r < 4; r++) u[q][r] = (a.U + r * a.plane + (int64_t)y * a.pitch)[x];
                shock[q] = a.shock ? (a.shock + (int64_t)y * a.nx)[x] : 0u;
            }
        };
        auto layer1 = [&](int row, NetRow& dst) {
#pragma unroll
            for (int q = 0; q < 3; q++) {
                f32x4 acc[2] = {f32x4{0.0f, 0.0f, 0.0f, 0.0f}, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
                for (int t = 0; t < 3; t++) {
                    const bf16x8 v = load8(img[(row + tap[t] / 3) & 3][16 * q + j + tap[t] % 3]);
                    const bf16x8 B = (4 * t + g < 9) ? v : zero8();
#pragma unroll
                    for (int mt = 0; mt < 2; mt++)
                        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[mt][t], B, acc[mt], 0, 0, 0);
                }
                finish(1, row, f0 + 16 * q, acc, bias, dst);
            }
        };
        auto layer5 = [&](int s, f32x4 (&acc)[3]) {
#pragma unroll
            for (int q = 0; q < 3; q++) acc[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int q = 0; q < 3; q++) {   // five segments: wave 7's last repeats its second
                    const int f = 8 + 16 * min(3 * h + q, NET_OUT / 16 - 1) + j;
                    const bf16x8 B = load8(buf[6 + ((s + 1 + t / 3) & 3)][g][f + t % 3]);
                    acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w5[t], B, acc[q], 0, 0, 0);
                }
        };
        auto put = [&](int row, const f32x4 (&acc)[3], const float (&u)[3][4], const uint32_t (&shock)[3]) {
#pragma unroll
            for (int q = 0; q < 3; q++) {
                const int x = X0 + 8 + 16 * (3 * h + q) + j;
                if (3 * h + q < NET_OUT / 16 && g == 0 && x < a.nx) output<MODE>(a, x, row, acc[q], b5, u[q], shock[q], nfb);
            }
        };
        float us[3][3][4];
        uint32_t sh[3][3];
        bf16x8 ahead[3];   // rows r1 + 2 to r1 + 4 of the padded image
#pragma unroll
        for (int r = 0; r < 2; r++) keep(yc - 4 + r, fetch(yc - 4 + r));
#pragma unroll
        for (int r = 0; r < 3; r++) ahead[r] = fetch(yc - 2 + r);
        fetch_state(yc - 12, us[0], sh[0]);
        for (int s0 = 0; s0 < steps; s0 += 3) {
#pragma unroll
            for (int ph = 0; ph < 3; ph++) {
                const int s = s0 + ph, r1 = yc - 4 + s, r5 = r1 - 8;
                keep(r1 + 2, ahead[ph]);
                ahead[ph] = fetch(r1 + 5);
                fetch_state(r5 + 1, us[(ph + 1) % 3], sh[(ph + 1) % 3]);
                const bool one = r1 < ye + 4, five = r5 >= yc && r5 < ye;
                f32x4 acc[3];
                if (one && five) {   // in one piece of code: the layers fill each other's waits
                    layer5(s, acc);   // first: its reads cannot pass layer 1's writes
                    layer1(r1, buf[s & 1]);
                    put(r5, acc, us[ph], sh[ph]);
                } else if (one) {
                    layer1(r1, buf[s & 1]);
                } else if (five) {
                    layer5(s, acc);
                    put(r5, acc, us[ph], sh[ph]);
                }
                lds_barrier();
            }
        }
    }
    if (MODE == NET_APPLY) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) nfb += __shfl_xor(nfb, off);
        if (lane == 0 && nfb) atomicAdd(a.fallback, nfb);
    }
}

// --------------------------------------------------------- data gradient --
// The gradient at a hidden layer's input: the convolution with the taps
// flipped and the channels swapped (the packed weights), times the ReLU mask of
// the stored activation.  One wave = one 16-pixel segment of a row, walking
// `rows` rows; operands and results lie as in k_net.
template <int CIN>
__global__ __launch_bounds__(256, 3) void k_conv_bwd(const ConvArgs a)
{
    constexpr int COUT = 32, MT = 2;
    constexpr int S = (9 * CIN / 8 + 3) / 4;
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4, j = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    const int nseg = a.nx >> 4;
    const int seg = wave % nseg;
    const int y0 = (wave / nseg) * a.rows;
    if (y0 >= a.ny) return;
    const int y1 = min(a.ny, y0 + a.rows);
    const int x = seg * 16 + j;
    const int W2 = a.nx + 2;

    bf16x8 wA[MT][S];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int s = 0; s < S; s++) wA[mt][s] = load8(a.wa + ((size_t)(mt * S + s) * 64 + lane) * 8);

    auto finish = [&](const int y, const f32x4 (&acc)[MT]) {
        const size_t pix = (size_t)(y + 1) * W2 + (x + 1);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const uint2 m = *reinterpret_cast<const uint2*>(a.mask + pix * COUT + 16 * mt + 4 * g);
            const uint32_t mv[4] = {m.x & 0xffffu, m.x >> 16, m.y & 0xffffu, m.y >> 16};
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = (mv[r] != 0u && mv[r] < 0x8000u) ? acc[mt][r] : 0.0f;
            uint2 pk;
            pk.x = pk_bf16(v[0], v[1]);
            pk.y = pk_bf16(v[2], v[3]);
            *reinterpret_cast<uint2*>(a.out + pix * COUT + 16 * mt + 4 * g) = pk;
        }
    };

    if (CIN == 32) {
        // The B operand of tap (dy, dx) at output row y is padded input row
        // y+dy+1 at column x+dx: each output row needs three input rows of
        // three column shifts, and each new row costs three loads.  Input
        // rows live in a ring of RING buffers named at compile time (the row
        // loop is unrolled by RING, so the window slides by renaming, not by
        // copying registers, which would wait for the loads): the loads of
        // row y+2+PF are issued while row y is computed, PF rows ahead of
        // their use, so the memory latency overlaps PF rows of MFMAs.
        constexpr int PF = 2, RING = 3 + PF;
        bf16x8 Rb[RING][3];
        auto load_row = [&](const int k, bf16x8 (&dst)[3]) {   // padded row y0 + k
            const int yr = min(y0 + k, a.ny + 1);
#pragma unroll
            for (int d = 0; d < 3; d++) dst[d] = load8(a.in + ((size_t)yr * W2 + (x + d)) * CIN + g * 8);
        };
#pragma unroll
        for (int k = 0; k < RING - 1; k++) load_row(k, Rb[k]);
        for (int base = y0; base < y1; base += RING) {
#pragma unroll
            for (int u = 0; u < RING; u++) {
                const int y = base + u;
                if (y < y1) {
                    load_row(y - y0 + RING - 1, Rb[(u + RING - 1) % RING]);
                    f32x4 acc[MT];
#pragma unroll
                    for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int t = 0; t < 9; t++)
#pragma unroll
                        for (int mt = 0; mt < MT; mt++)
                            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wA[mt][t], Rb[(u + t / 3) % RING][t % 3],
                                                                             acc[mt], 0, 0, 0);
                    finish(y, acc);
                }
            }
        }
    } else {
        for (int y = y0; y < y1; y++) {
            f32x4 acc[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < S; s++) {
                int tap = 4 * s + g;
                const bool valid = tap < 9;
                tap = valid ? tap : 8;
                const int dy = tap / 3 - 1, dx = tap % 3 - 1;
                bf16x8 B = load8(a.in + ((size_t)(y + 1 + dy) * W2 + (x + 1 + dx)) * CIN);
                B = valid ? B : zero8();
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wA[mt][s], B, acc[mt], 0, 0, 0);
            }
            finish(y, acc);
        }
    }
}

// ---------------------------------------------------------- weight gradient --
// dW[tap][ci][co] = sum_p a[p + tap][ci] * gz[p][co],  db[co] = sum_p gz[p][co].
// A workgroup owns a 64-pixel column strip over `rows` rows.  Per output row
// it stages gz (channel-major, gT[co][px]) and one new input row in LDS,
// channel-major and shifted by each dx (aT[slot][dx][ci][px] =
// a[row][x0+px+dx][ci]); the three input rows a tap can reach live in a ring
// of three slots, so each input row is staged once.  Each lane's 8
// consecutive pixels of one channel are then one aligned 16-byte LDS read.
// The pixels are the MFMA reduction dimension: A = gz^T (rows = co), B =
// shifted input (columns = ci).  A row's A operands are read once per wave; a
// wave owns a fixed set of (tap, ci tile) pairs, reads each pair's B operand
// once for all co tiles, and wave 3 also multiplies A by ones, which gives db;
// partial sums go to part[workgroup].
// Bound by the LDS round of a row (staging, barrier, operand reads).
constexpr int LPX = 72;   // LDS row pitch in elements (64 pixels + 8 padding)

// All layers in one launch, which needs every layer's gradient image kept: a
// launch per layer of a small image fills the chip only with two rows per
// workgroup, which stages as many again and leaves four times the partials.
// 256^2, the five layers and their reduction: 64 + 13 us as five launches (44.6
// for one 32 -> 32 layer with 16 rows, two operand reads per product and db
// summed by threads), now 29 + 5; a training step at 1024^2 0.805 -> 0.726 ms
// against the same kernels layer by layer, although the data gradients, back to
// back, then miss the cache (1024^2: 49 -> 58 us, 31 -> 47 the last).
constexpr int WGRAD_FILL = 384;
constexpr int WGRAD_LDS = (9 * 32 + 32) * LPX;

template <int CI, int CO>
__device__ __forceinline__ void wgrad(const WgradLayer& a, int wg, int nx, int ny, int rows, uint16_t* lds)
{
    constexpr int CIL = CI < 16 ? 16 : CI;
    constexpr int COL = CO < 16 ? 16 : CO;
    constexpr int MT = COL / 16, NT = CIL / 16;
    constexpr int PAIRS = 9 * NT;
    constexpr int NPW = (PAIRS + 3) / 4;
    uint16_t (*const aT)[3][CIL][LPX] = reinterpret_cast<uint16_t (*)[3][CIL][LPX]>(lds);
    uint16_t (*const gT)[LPX] = reinterpret_cast<uint16_t (*)[LPX]>(lds + 9 * CIL * LPX);
    static_assert((9 * CIL + COL) * LPX <= WGRAD_LDS, "LDS of a workgroup");

    const int tid = threadIdx.x;
    const int lane = tid & 63, g = lane >> 4, j = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nstrip = nx >> 6;
    const int x0 = (wg % nstrip) * 64;
    const int y0 = (wg / nstrip) * rows;
    const int y1 = min(ny, y0 + rows);
    const int W2 = nx + 2;

    // zero the padding channels once (never written below)
    if (CIL > CI)
        for (int i = tid; i < 9 * (CIL - CI) * LPX; i += 256) {
            const int t = i / ((CIL - CI) * LPX), rem = i % ((CIL - CI) * LPX);
            aT[t / 3][t % 3][CI + rem / LPX][rem % LPX] = 0;
        }
    if (COL > CO)
        for (int i = tid; i < (COL - CO) * LPX; i += 256) gT[CO + i / LPX][i % LPX] = 0;

    // input row r (interior index, -1 <= r <= ny) into ring slot (r + 3) % 3
    auto stage_row = [&](int r) {
        const int slot = (r + 3) % 3;
        for (int i = tid; i < 66 * (CI / 8); i += 256) {
            const int ps = i / (CI / 8) - 1, cb = i % (CI / 8);
            const uint4 v = *reinterpret_cast<const uint4*>(a.a + ((size_t)(r + 1) * W2 + x0 + ps + 1) * CI + cb * 8);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int dxi = 0; dxi < 3; dxi++) {
                const int px = ps - (dxi - 1);
                if (px >= 0 && px < 64) {
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        aT[slot][dxi][cb * 8 + e][px] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
                }
            }
        }
    };

    f32x4 acc[NPW][MT], db[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        db[mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < NPW; u++) acc[u][mt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const uint4 one4 = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
    const bf16x8 ones = __builtin_bit_cast(bf16x8, one4);

    stage_row(y0 - 1);
    stage_row(y0);
    for (int y = y0; y < y1; y++) {
        __syncthreads();
        for (int i = tid; i < 64 * (CO / 8); i += 256) {
            const int px = i / (CO / 8), cb = i % (CO / 8);
            const uint4 v = *reinterpret_cast<const uint4*>(a.gz + ((size_t)(y + 1) * W2 + x0 + px + 1) * CO + cb * 8);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 8; e++) gT[cb * 8 + e][px] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
        }
        stage_row(y + 1);
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            bf16x8 A[MT];
#pragma unroll
            for (int mt = 0; mt < MT; mt++) A[mt] = load8(&gT[16 * mt + j][32 * ks + 8 * g]);
#pragma unroll
            for (int u = 0; u < NPW; u++) {
                const int q = wave + 4 * u;
                if (q < PAIRS) {
                    const int tap = q % 9, nt = q / 9;
                    const int slot = (y + tap / 3 + 2) % 3;   // input row y + dy, dy = tap/3 - 1
                    const bf16x8 B = load8(&aT[slot][tap % 3][16 * nt + j][32 * ks + 8 * g]);
#pragma unroll
                    for (int mt = 0; mt < MT; mt++)
                        acc[u][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[mt], B, acc[u][mt], 0, 0, 0);
                }
            }
            if (wave == 3)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
                    db[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[mt], ones, db[mt], 0, 0, 0);
        }
    }

    float* P = a.part + (size_t)wg * (9 * CI * CO + CO);
#pragma unroll
    for (int u = 0; u < NPW; u++) {
        const int q = wave + 4 * u;
        if (q < PAIRS) {
            const int tap = q % 9, ci = 16 * (q / 9) + j;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int co = 16 * mt + 4 * g + r;
                    if (co < CO && ci < CI) P[((size_t)tap * CI + ci) * CO + co] = acc[u][mt][r];
                }
        }
    }
    if (wave == 3 && j == 0)   // every column holds the sum
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int co = 16 * mt + 4 * g + r;
                if (co < CO) P[9 * CI * CO + co] = db[mt][r];
            }
}

__global__ __launch_bounds__(256) void k_wgrad(const WgradArgs a)
{
    __shared__ __attribute__((aligned(16))) uint16_t lds[WGRAD_LDS];
    const WgradLayer& l = a.layer[blockIdx.x / a.nwg];
    const int wg = (int)(blockIdx.x % a.nwg);
    if (l.ci == 8) wgrad<8, 32>(l, wg, a.nx, a.ny, a.rows, lds);
    else if (l.co == 8) wgrad<32, 8>(l, wg, a.nx, a.ny, a.rows, lds);
    else wgrad<32, 32>(l, wg, a.nx, a.ny, a.rows, lds);
}

// ------------------------------------------------------------------ helpers --
__device__ __forceinline__ float pressure(const float* U, int64_t plane, float gamma)
{
    const float r = U[0], mu = U[plane], mv = U[2 * plane], E = U[3 * plane];
    return (gamma - 1.0f) * (E - 0.5f * (mu * mu + mv * mv) / r);
}

__global__ __launch_bounds__(256) void k_pack(const PackArgs a)
{
    const int x = blockIdx.x * 256 + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= a.nx) return;
    const float* U = a.U + (size_t)y * a.pitch + x;
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = (U[r * a.plane] - a.mean[r]) * a.iscale[r];
    uint4 pk;
    pk.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
    pk.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
    pk.z = 0u;
    pk.w = 0u;
    *reinterpret_cast<uint4*>(a.X + ((size_t)(y + 1) * (a.nx + 2) + x + 1) * 8) = pk;
    if (a.shock) {
        // normalised second difference of the pressure, the larger of x and y
        const int xl = x > 0 ? -1 : 0, xr = x < a.nx - 1 ? 1 : 0;
        const int yd = y > 0 ? -a.pitch : 0, yu = y < a.ny - 1 ? a.pitch : 0;
        const float p = pressure(U, a.plane, a.gamma);
        const float pl = pressure(U + xl, a.plane, a.gamma), pr = pressure(U + xr, a.plane, a.gamma);
        const float pd = pressure(U + yd, a.plane, a.gamma), pu = pressure(U + yu, a.plane, a.gamma);
        const float sx = fabsf(pr - 2.0f * p + pl) / (pr + 2.0f * p + pl);
        const float sy = fabsf(pu - 2.0f * p + pd) / (pu + 2.0f * p + pd);
        a.shock[(size_t)y * a.nx + x] = (sx > a.theta || sy > a.theta || !(sx == sx) || !(sy == sy)) ? 1 : 0;
    }
}

__global__ __launch_bounds__(256) void k_loss(const LossArgs a)
{
    __shared__ float red[256];
    const int64_t np = (int64_t)a.nx * a.ny;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    float l = 0.0f;
    if (i < np) {
        const int y = (int)(i / a.nx), x = (int)(i % a.nx);
        float gv[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float t = (a.T[r * np + i] - a.Uc[r * np + i]) * a.inv_scale[r];
            const float d = a.Y[r * np + i] - t;
            l += d * d;
            gv[r] = a.gscale * 2.0f * d;
        }
        uint4 pk;
        pk.x = (uint32_t)f2bf(gv[0]) | ((uint32_t)f2bf(gv[1]) << 16);
        pk.y = (uint32_t)f2bf(gv[2]) | ((uint32_t)f2bf(gv[3]) << 16);
        pk.z = 0u;
        pk.w = 0u;
        *reinterpret_cast<uint4*>(a.G + ((size_t)(y + 1) * (a.nx + 2) + x + 1) * 8) = pk;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) a.part[blockIdx.x] = red[0];
}

// Sums of the weight gradients' workgroup partials, every layer in one launch:
// a workgroup adds 64 consecutive entries of one layer, its 16 waves interleaved
// subsets of the partials, combined in a fixed order, and writes the layer's
// real layout W[9][ci_r][co_r] followed by b[co_r] (padding channels dropped);
// the last workgroup sums the loss.  Bound by the partials' bytes.  Ten
// launches (two per layer) took 50 us of a 256^2 gradient, one 13, with
// wgrad_rows()'s longer workgroups 5 (and the loss 3.7 in a launch of its own).
__global__ __launch_bounds__(1024) void k_reduce_grad(const ReduceArgs a)
{
    __shared__ float red[16][64];
    if (blockIdx.x == gridDim.x - 1) {
        float* const sum = red[0];
        float s = 0.0f;
        if (threadIdx.x < 256)
            for (int i = threadIdx.x; i < a.nloss; i += 256) s += a.lossp[i];
        sum[threadIdx.x] = s;
        for (int k = 128; k > 0; k >>= 1) {
            __syncthreads();
            if ((int)threadIdx.x < k) sum[threadIdx.x] += sum[threadIdx.x + k];
        }
        if (threadIdx.x == 0) a.loss[0] = sum[0] * a.loss_scale;
        return;
    }
    int l = 0;
    while (l + 1 < a.nlayers && (int)blockIdx.x >= a.layer[l + 1].first) l++;
    const ReduceLayer L = a.layer[l];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int stride = 9 * L.ci * L.co + L.co;
    const int s = ((int)blockIdx.x - L.first) * 64 + tx;
    float acc = 0.0f;
    if (s < stride)
        for (int w = ty; w < L.nparts; w += 16) acc += L.part[(size_t)w * stride + s];
    red[ty][tx] = acc;
    __syncthreads();
    if (ty != 0 || s >= stride) return;
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; k++) v += red[k][tx];
    int dst = -1;
    if (s < 9 * L.ci * L.co) {
        const int tap = s / (L.ci * L.co), rem = s % (L.ci * L.co);
        const int ci = rem / L.co, co = rem % L.co;
        if (ci < L.ci_r && co < L.co_r) dst = (tap * L.ci_r + ci) * L.co_r + co;
    } else {
        const int co = s - 9 * L.ci * L.co;
        if (co < L.co_r) dst = 9 * L.ci_r * L.co_r + co;
    }
    if (dst >= 0) L.grads[dst] = v;
}

__global__ __launch_bounds__(256) void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                                              float* __restrict__ v, int n, float lr, float b1, float b2, float eps,
                                              float c1, float c2)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

template <int CIN, int COUT>
__global__ __launch_bounds__(256) void k_pack_w(const float* __restrict__ W, int ci_r, int co_r, int transposed,
                                                uint16_t* __restrict__ wa)
{
    constexpr int MT = (COUT + 15) / 16;
    constexpr int S = (9 * CIN / 8 + 3) / 4;
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= MT * S * 64 * 8) return;
    const int e = idx & 7, lane = (idx >> 3) & 63;
    const int s = (idx >> 9) % S, mt = (idx >> 9) / S;
    const int o = 16 * mt + (lane & 15), g = lane >> 4;
    int tap, i;
    if (CIN == 32) {
        tap = s;
        i = 8 * g + e;
    } else {
        tap = 4 * s + g;
        i = e;
    }
    float val = 0.0f;
    if (tap < 9) {
        if (!transposed) {
            if (o < co_r && i < ci_r) val = W[((size_t)tap * ci_r + i) * co_r + o];
        } else {
            if (o < ci_r && i < co_r) val = W[((size_t)(8 - tap) * ci_r + o) * co_r + i];
        }
    }
    wa[idx] = f2bf(val);
}

__global__ __launch_bounds__(256) void k_state_copy(const float* __restrict__ src, int64_t splane, int spitch,
                                                    float* __restrict__ dst, int64_t dplane, int dpitch, int nx)
{
    const int x = blockIdx.x * 256 + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= nx) return;
#pragma unroll
    for (int r = 0; r < 4; r++) dst[r * dplane + (size_t)y * dpitch + x] = src[r * splane + (size_t)y * spitch + x];
}

__global__ __launch_bounds__(256) void k_restrict2(const float* __restrict__ U, int64_t plane, int pitch, int nxc,
                                                   int nyc, float* __restrict__ dst)
{
    const int x = blockIdx.x * 256 + threadIdx.x;
    const int y = blockIdx.y;
    if (x >= nxc) return;
    const size_t np = (size_t)nxc * nyc;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float* u = U + r * plane + (size_t)(2 * y) * pitch + 2 * x;
        dst[r * np + (size_t)y * nxc + x] = 0.25f * ((u[0] + u[1]) + (u[pitch] + u[pitch + 1]));
    }
}

// ---------------------------------------------------------------- launchers --
hipError_t launch_net(NetArgs a, int mode, hipStream_t s)
{
    // one workgroup fills a CU: rows so that one round of the 256 CUs takes the
    // image, at least 4 (a strip's steps are its rows and 12 more)
    const int nstrip = (a.nx + NET_OUT - 1) / NET_OUT;
    const int chunks = nstrip < 256 ? 256 / nstrip : 1;
    a.rows = (a.ny + chunks - 1) / chunks;
    if (a.rows < 4) a.rows = 4;
    if (a.rows > 128) a.rows = 128;
    const dim3 grid(nstrip * ((a.ny + a.rows - 1) / a.rows));
    if (mode == NET_APPLY) hipLaunchKernelGGL((k_net<NET_APPLY, false>), grid, dim3(512), 0, s, a);
    else if (a.act[0]) hipLaunchKernelGGL((k_net<NET_OUT_PLANES, true>), grid, dim3(512), 0, s, a);
    else hipLaunchKernelGGL((k_net<NET_OUT_PLANES, false>), grid, dim3(512), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_conv_bwd(int cin, const ConvArgs& a, hipStream_t s)
{
    const int waves = (a.nx / 16) * ((a.ny + a.rows - 1) / a.rows);
    const dim3 grid((waves + 3) / 4);
    if (cin == 8) hipLaunchKernelGGL((k_conv_bwd<8>), grid, dim3(256), 0, s, a);
    else if (cin == 32) hipLaunchKernelGGL((k_conv_bwd<32>), grid, dim3(256), 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

// Rows per workgroup: the most, up to 16, with which the layers together still
// make WGRAD_FILL workgroups (at least 2 rows: every workgroup stages two
// more).  256^2, sums and reduction: 384 workgroups 29 + 5 us, 768 31 + 8, 1536
// 38 + 13; 128^2, 512^2 and 1024^2 the same with each.
static int wgrad_rows(int nx, int ny)
{
    int rows = 16;
    while (rows > 2 && MAX_LAYERS * (int64_t)(nx / 64) * ((ny + rows - 1) / rows) < WGRAD_FILL) rows /= 2;
    return rows;
}
int wgrad_workgroups(int nx, int ny)
{
    const int rows = wgrad_rows(nx, ny);
    return (nx / 64) * ((ny + rows - 1) / rows);
}

hipError_t launch_wgrad(WgradArgs a, hipStream_t s)
{
    for (int l = 0; l < a.nlayers; l++) {
        const int ci = a.layer[l].ci, co = a.layer[l].co;
        if (!((ci == 8 && co == 32) || (ci == 32 && co == 32) || (ci == 32 && co == 8))) return hipErrorInvalidValue;
    }
    a.rows = wgrad_rows(a.nx, a.ny);
    a.nwg = wgrad_workgroups(a.nx, a.ny);
    hipLaunchKernelGGL(k_wgrad, dim3((unsigned)a.nlayers * a.nwg), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_pack(const PackArgs& a, hipStream_t s)
{
    hipLaunchKernelGGL(k_pack, dim3((a.nx + 255) / 256, a.ny), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_loss(const LossArgs& a, int* nblocks, hipStream_t s)
{
    const int64_t np = (int64_t)a.nx * a.ny;
    const int n = (int)((np + 255) / 256);
    *nblocks = n;
    hipLaunchKernelGGL(k_loss, dim3(n), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_reduce_grad(ReduceArgs a, hipStream_t s)
{
    int blocks = 0;
    for (int l = 0; l < a.nlayers; l++) {
        a.layer[l].first = blocks;
        blocks += (9 * a.layer[l].ci * a.layer[l].co + a.layer[l].co + 63) / 64;
    }
    hipLaunchKernelGGL(k_reduce_grad, dim3(blocks + 1), dim3(1024), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_adam(float* w, const float* g, float* m, float* v, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2, hipStream_t s)
{
    hipLaunchKernelGGL(k_adam, dim3((n + 255) / 256), dim3(256), 0, s, w, g, m, v, n, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}

int packed_weight_elems(int cin, int cout) { return ((cout + 15) / 16) * ((9 * cin / 8 + 3) / 4) * 64 * 8; }

hipError_t launch_pack_weights(int cin, int cout, const float* W, int ci_r, int co_r, int transposed, uint16_t* wa,
                               hipStream_t s)
{
    const int n = packed_weight_elems(cin, cout);
    const dim3 grid((n + 255) / 256);
    if (cin == 8 && cout == 32) hipLaunchKernelGGL((k_pack_w<8, 32>), grid, dim3(256), 0, s, W, ci_r, co_r, transposed, wa);
    else if (cin == 32 && cout == 32)
        hipLaunchKernelGGL((k_pack_w<32, 32>), grid, dim3(256), 0, s, W, ci_r, co_r, transposed, wa);
    else if (cin == 32 && cout == 8)
        hipLaunchKernelGGL((k_pack_w<32, 8>), grid, dim3(256), 0, s, W, ci_r, co_r, transposed, wa);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_state_copy(const float* src, int64_t splane, int spitch, float* dst, int64_t dplane, int dpitch,
                             int nx, int ny, hipStream_t s)
{
    hipLaunchKernelGGL(k_state_copy, dim3((nx + 255) / 256, ny), dim3(256), 0, s, src, splane, spitch, dst, dplane,
                       dpitch, nx);
    return hipGetLastError();
}

hipError_t launch_restrict2(const float* U, int64_t plane, int pitch, int nxc, int nyc, float* dst, hipStream_t s)
{
    hipLaunchKernelGGL(k_restrict2, dim3((nxc + 255) / 256, nyc), dim3(256), 0, s, U, plane, pitch, nxc, nyc, dst);
    return hipGetLastError();
}

}  // namespace hfn
