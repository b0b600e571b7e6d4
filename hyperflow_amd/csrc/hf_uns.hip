// hf_uns.hip -- gfx950 kernels of the unstructured quadrilateral-cell
// Godunov solver (src/fvm_2d_uns), FP64, bit-exact with the reference:
// compiled with -ffp-contract=off, every expression in the reference's order.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "hf_common.h"
#include "hf_physics.h"
#include "hf_uns.h"

namespace hfu {

using hf::MathF64;
typedef double R;

__device__ __forceinline__ unsigned long long bits_of(double d) { return (unsigned long long)__double_as_longlong(d); }
__device__ __forceinline__ double double_of(unsigned long long b) { return __longlong_as_double((long long)b); }

// EulerIdealGasModel::rotate_flow_values (model/euler_ideal_gas/euler_ideal_gas.cpp:152-164)
__device__ __forceinline__ void rotate(double c, double s, const double W[4], double Rv[4])
{
    Rv[0] = W[0];
    Rv[1] = c * W[1] + s * W[2];
    Rv[2] = -1.0 * s * W[1] + c * W[2];
    Rv[3] = W[3];
}

// TimeStep::operator()'s per-cell quotient (scheme/timestep/timestep.cpp:41-52)
__device__ __forceinline__ double cell_dt(const double U[4], double dr, double gamma, double g1)
{
    double u, v, p, E;
    hf::prims<MathF64>(U[0], U[1], U[2], U[3], g1, u, v, p, E);
    const double a = hf::sound<MathF64>(gamma, p, U[0]);
    return dr / (__builtin_fabs(__builtin_sqrt(u * u + v * v)) + a);
}

// minimum over the wave of bit patterns (positive doubles order like their bits;
// NaN patterns are larger than every number, as std::min ignores NaN quotients)
__device__ __forceinline__ unsigned long long wave_min_bits(unsigned long long b)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(b, off);
        b = o < b ? o : b;
    }
    return b;
}

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  The grid is padded to a multiple of 8 and workgroup b works on cell
// chunk (b % 8) * (grid / 8) + b / 8, so each XCD sweeps one contiguous
// eighth of the cells and finds most neighbour states in its own L2.
constexpr int XCDS = 8;
__device__ __forceinline__ int cell_chunk()
{
    return (int)(blockIdx.x % XCDS) * (int)(gridDim.x / XCDS) + (int)(blockIdx.x / XCDS);
}
inline dim3 chunk_grid(int n) { return dim3((unsigned)(((n + 255) / 256 + XCDS - 1) / XCDS * XCDS)); }

// The workgroup's minimum into one way of a slot: wave minima through LDS,
// then one atomic.  Called by every thread of the workgroup.
__device__ __forceinline__ void block_min_to_slot(unsigned long long cand, unsigned long long* slot)
{
    __shared__ unsigned long long wmin[4];
    cand = wave_min_bits(cand);
    if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = cand;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long b = wmin[0];
        for (int w = 1; w < 4; w++) b = wmin[w] < b ? wmin[w] : b;
        atomicMin(slot + (blockIdx.x % SLOT_WAYS) * SLOT_STRIDE, b);
    }
}

// The general division and root (QUICK false) or those of hf::q64, whose
// range the rotated states are checked against: their masks gather in bad.
template <bool QUICK>
struct Face;
template <>
struct Face<false> {
    typedef hf::State<R> State;
    static __device__ __forceinline__ State state(const double U[4], double gamma, double g1, double, hf::q64::mask&,
                                                  const hf::q64::Limits&)
    {
        return hf::make_state<MathF64>(U, gamma, g1);
    }
    static __device__ __forceinline__ void hllc(const State& L, const State& Rs, double F[4], hf::q64::mask&,
                                                const hf::q64::Limits&)
    {
        hf::hllc<MathF64, true>(L, Rs, F);
    }
    static __device__ __forceinline__ double dt(const double U[4], double dr, double gamma, double g1, hf::q64::mask&,
                                                const hf::q64::Limits&)
    {
        return cell_dt(U, dr, gamma, g1);
    }
};
template <>
struct Face<true> {
    typedef hf::q64::State State;
    static __device__ __forceinline__ State state(const double U[4], double gamma, double g1, double ig1,
                                                  hf::q64::mask& bad, const hf::q64::Limits& lim)
    {
        bad |= hf::q64::out_of_range(U, lim);
        return hf::q64::make_state(U, gamma, g1, ig1, bad, lim);
    }
    static __device__ __forceinline__ void hllc(const State& L, const State& Rs, double F[4], hf::q64::mask& bad,
                                                const hf::q64::Limits& lim)
    {
        hf::q64::hllc<true>(L, Rs, F, bad, lim);
    }
    // A momentum too small for the quotient leaves a speed far below the last
    // bit of the sound speed; at rest the root of zero is set apart.  A NaN in
    // the new state, a pressure of zero or below make the sum NaN.
    static __device__ __forceinline__ double dt(const double U[4], double dr, double gamma, double g1,
                                                hf::q64::mask& bad, const hf::q64::Limits& lim)
    {
        const double y = hf::q64::rcp(U[0]);
        const double u = hf::q64::div_pos(U[1], U[0], y), v = hf::q64::div_pos(U[2], U[0], y);
        const double q2 = u * u + v * v;
        const double p = g1 * hf::q64::fma(-0.5, U[0] * q2, U[3]);
        const double speed = q2 == 0.0 ? 0.0 : hf::q64::sqrt(q2);
        const double d = speed + hf::q64::sqrt(hf::q64::div_pos(gamma * p, U[0], y));
        bad |= __ballot(!(U[0] >= lim.low)) | __ballot(!(U[3] >= lim.low)) | __ballot(!(d == d)) |
               __ballot(!(dr >= 0x1p-200)) | __ballot(!(dr <= 0x1p200));
        return hf::q64::div_pos(dr, d, hf::q64::rcp(d));
    }
};

// GodunovScheme::operator() (scheme/godunov/godunov.cpp:31-77), boundary
// states of BoundaryConditions (scheme/boundary/boundary.cpp:29-69), and
// ForwardEulerODESolver (scheme/ode/forward_euler/forward_euler.cpp:16-30) of
// one cell: its new state and its term of the next dt.  Returns the lanes out
// of range (QUICK).
template <bool QUICK>
__device__ __forceinline__ hf::q64::mask advance_cell(const UnsMesh& m, const UnsStep& s, int c, const double U[4],
                                                      double dt, double N[4], double& term)
{
    typedef Face<QUICK> Fc;
    const int n = m.n;
    const double gamma = m.gamma, g1 = m.gamma - 1.0;
    const double ig1 = QUICK ? 1.0 / g1 : 0.0;
    const hf::q64::Limits lim;
    hf::q64::mask bad = 0;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    double shortest = 1e16;
#pragma unroll 1   // see k_uns_step
    for (int e = 0; e < 4; e++) {
        const int nb = m.nbr[(size_t)e * n + c];
        const int ct = m.cs_terms;
        const double cr = m.cs[(size_t)(ct * e + 0) * n + c], sr = m.cs[(size_t)(ct * e + 1) * n + c];
        double cb = cr, sb = -sr;   // the back rotation mirrors the forward one (checked on the host)
        if (ct == 4) {
            cb = m.cs[(size_t)(4 * e + 2) * n + c];
            sb = m.cs[(size_t)(4 * e + 3) * n + c];
        }
        double V[4];
        if (nb >= 0) {
#pragma unroll
            for (int k = 0; k < 4; k++) V[k] = s.A[(size_t)k * n + nb];
        } else if (nb == -1) {   // reflective (boundary.cpp:48-56)
            double t[4];
            rotate(cr, sr, U, t);
            t[1] *= -1.0;
            rotate(cb, sb, t, V);
        } else if (nb == -2) {   // transmissive
#pragma unroll
            for (int k = 0; k < 4; k++) V[k] = U[k];
        } else {                 // inlet
#pragma unroll
            for (int k = 0; k < 4; k++) V[k] = m.inlet[k];
        }
        double rU[4], rV[4], F[4], f[4];
        rotate(cr, sr, U, rU);
        rotate(cr, sr, V, rV);
        const typename Fc::State L = Fc::state(rU, gamma, g1, ig1, bad, lim);
        const typename Fc::State Rs = Fc::state(rV, gamma, g1, ig1, bad, lim);
        Fc::hllc(L, Rs, F, bad, lim);
        rotate(cb, sb, F, f);
        const double len = m.len[(size_t)e * n + c];
        shortest = (shortest < len) ? shortest : len;   // Polygon's incircle radius (polygon.cpp:79-91)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            f[k] *= len;
            acc[k] += f[k];
        }
    }
    const double iv = m.inv_vol[c];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        double x = acc[k];
        x *= iv;
        x *= -1.0;
        x *= dt;
        x += U[k];
        N[k] = x;
    }
    term = Fc::dt(N, shortest, gamma, g1, bad, lim);
    return bad;
}

// One step.  A wave runs hf::q64's arithmetic and, where a lane is out of its
// range, the general one over it.
// Bound by FP64 arithmetic: 274 VALU instructions per edge, 6 of them
// quarter-rate (362 and 14 by the general one), with the edges in a loop so
// that four waves per SIMD keep their registers (108; unrolled, the edges'
// values are spilled at four waves, and at two or three waves, where they fit,
// a step takes 27 and 29 us).  The memory side alone (184 bytes a cell) takes
// 14.2 us, the arithmetic alone 19.8.  367 500 cells: 27.1 -> 22.3 us a step,
// 20.9 with the state requested ahead of the dt's reduction (the figures below
// are against 22.3 but the last).
// Not faster: an edge's reads requested an edge ahead (22.1-23.2), a wave per
// edge and 64 cells per workgroup (23.7), one-wave workgroups (22.8), five
// waves per SIMD (25.6, 8 registers spilled), the first edge's neighbour requested
// beside the state (21.2 against 20.9).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_uns_step(const UnsMesh m,
                                                                                          const UnsStep s)
{
    const int c = cell_chunk() * 256 + threadIdx.x;
    const int n = m.n;
    const int lane = threadIdx.x & 63;
    unsigned long long slot = 0ull;
    if (!s.use_fixed) slot = s.slots[s.rd * SLOT_WORDS + lane * SLOT_STRIDE];
    double U[4];   // on its way while the dt is reduced (21.4 -> 20.9 us at 367 500 cells)
#pragma unroll
    for (int k = 0; k < 4; k++) U[k] = s.A[(size_t)k * n + (c < n ? c : n - 1)];
    double dt;
    const long long kcall = s.kdev ? (long long)s.kdev[s.kpar] + 1 : s.kcall;
    if (s.use_fixed) {
        dt = s.fixed_dt;
    } else {
        const double cf = (kcall <= 10) ? 0.2 * m.cfl : m.cfl;   // timestep.cpp:57-61
        dt = cf * double_of(wave_min_bits(slot));
    }
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        if (threadIdx.x == 0 && s.kdev) s.kdev[s.kpar ^ 1] = (unsigned long long)kcall;
        if (threadIdx.x == 0 && !s.use_fixed && kcall >= 1 && kcall <= s.hist_cap) s.hist[kcall - 1] = dt;
        if (s.rs >= 0) s.slots[s.rs * SLOT_WORDS + lane * SLOT_STRIDE] = SLOT_EMPTY;
    }
    unsigned long long cand = ~0ull;
    if (c < n) {
        double N[4], term;
        // density and energy, which the rotations leave alone, before arithmetic
        // that would be done twice: out of range a step of 367 500 cells takes 25.0
        // us, 38.6 if the edges find it
        // by their high words: q64's bounds are powers of two (2^-60 and 2^40)
        constexpr unsigned LOW = (1023u - 60u) << 20, HIGH = (1023u + 40u) << 20;
        const unsigned r = (unsigned)__double2hiint(U[0]) - LOW, E = (unsigned)__double2hiint(U[3]) - LOW;
        hf::q64::mask bad = __ballot((r > E ? r : E) > HIGH - LOW);
        if (!bad && hf::q64::constants_in_range(m.gamma, m.gamma - 1.0))
            bad = advance_cell<true>(m, s, c, U, dt, N, term);
        else
            bad = 1;
        if (bad) advance_cell<false>(m, s, c, U, dt, N, term);
#pragma unroll
        for (int k = 0; k < 4; k++) s.B[(size_t)k * n + c] = N[k];
        cand = bits_of(term);
    }
    if (s.wr >= 0) block_min_to_slot(cand, s.slots + s.wr * SLOT_WORDS);
}

__global__ __launch_bounds__(256) void k_uns_scan(const UnsMesh m, const double* __restrict__ A,
                                                  unsigned long long* slot)
{
    const int c = cell_chunk() * 256 + threadIdx.x;
    const int n = m.n;
    unsigned long long cand = ~0ull;
    if (c < n) {
        double U[4];
#pragma unroll
        for (int k = 0; k < 4; k++) U[k] = A[(size_t)k * n + c];
        double shortest = 1e16;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const double len = m.len[(size_t)e * n + c];
            shortest = (shortest < len) ? shortest : len;
        }
        cand = bits_of(cell_dt(U, shortest, m.gamma, m.gamma - 1.0));
    }
    block_min_to_slot(cand, slot);
}

__global__ void k_uns_reset(unsigned long long* slot) { slot[threadIdx.x * SLOT_STRIDE] = SLOT_EMPTY; }

hipError_t launch_uns_step(const UnsMesh& m, const UnsStep& s, hipStream_t st, hipEvent_t e0, hipEvent_t e1)
{
    if (e0 || e1) hipExtLaunchKernelGGL(k_uns_step, chunk_grid(m.n), dim3(256), 0, st, e0, e1, 0, m, s);
    else hipLaunchKernelGGL(k_uns_step, chunk_grid(m.n), dim3(256), 0, st, m, s);
    return hipGetLastError();
}

hipError_t launch_uns_scan(const UnsMesh& m, const double* A, unsigned long long* slots, int slot, hipStream_t st)
{
    hipLaunchKernelGGL(k_uns_reset, dim3(1), dim3(SLOT_WAYS), 0, st, slots + slot * SLOT_WORDS);
    hipLaunchKernelGGL(k_uns_scan, chunk_grid(m.n), dim3(256), 0, st, m, A, slots + slot * SLOT_WORDS);
    return hipGetLastError();
}

}  // namespace hfu
