// hf_kernels.h -- gfx950 kernels of the block-Cartesian Euler step.
//
// Update kernels ("sweeps"): each 64-lane wave owns a strip of padded columns
// (lane l <-> column x0+l) and walks down `rows` output rows of one block.
// The reconstruction window, face states, both HLLC fluxes and the update of
// a row live in registers; x neighbours come from cross-lane shuffles, y
// neighbours from the previous iteration.  Every conserved value is read once
// from HBM (plus the 2-lane halo at each strip edge and 2 halo rows per
// strip) and every output written once; nothing intermediate goes to memory.
// The new state's max wave speeds (for the next dt) are reduced in the same
// pass: wave shuffles, then a 64-bit atomic max per wave (store_maxima).
//
// The interior is read from A and the filled ghosts from G (the ghost fill
// writes them into the destination buffer), or ghosts are read from A where
// they mirror to (Lines), so no launch ever reads a cell that another wave of
// the same step writes.
#pragma once
#include <hip/hip_runtime.h>

#include "hf_common.h"
#include "hf_physics.h"

namespace hf {

template <class R>
__device__ __forceinline__ void load_cell(const R* __restrict__ base, int64_t plane, R u[4])
{
    u[0] = base[0];
    u[1] = base[plane];
    u[2] = base[2 * plane];
    u[3] = base[3 * plane];
}

// Whole-wave lane shifts by one lane through DPP (wave_shr:1 / wave_shl:1):
// lane l receives lane l-1 (up) or lane l+1 (down); the end lane, a halo lane
// in every sweep, receives zero (to keep its own value would take a move ahead
// of every shift).  No LDS round trip, unlike a bpermute shuffle.
__device__ __forceinline__ int dpp_up(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ int dpp_dn(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ double shfl_up1(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = dpp_up((int)(b & 0xffffffffll)), hi = dpp_up((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double shfl_dn1(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = dpp_dn((int)(b & 0xffffffffll)), hi = dpp_dn((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ float shfl_up1(float x) { return __int_as_float(dpp_up(__float_as_int(x))); }
__device__ __forceinline__ float shfl_dn1(float x) { return __int_as_float(dpp_dn(__float_as_int(x))); }

// Work items of a persistent launch: wave w first takes item w (no atomic, so
// a launch does not open with every wave hitting one counter), then tickets
// from the queue counter, offset by the number of waves.  Every
// lane executes the atomic (only lane 0 adds 1) so that no lane-divergent
// region surrounds the loop's exit test; lane 0's old value is the wave's
// ticket.  A lane-0-only branch here let the compiler's control-flow
// structurizer keep lanes 1..63 in the loop after lane 0 left it.
// (the last workgroup of a mirrored launch, `extra`, takes none)
__device__ __forceinline__ unsigned total_waves(unsigned extra = 0) { return (gridDim.x - extra) * (blockDim.x >> 6); }
__device__ __forceinline__ unsigned wave_id()
{
    // wave-uniform, but derived from threadIdx: say so, or the whole item loop
    // is compiled as divergent (vector loads of the item and block records)
    return __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
}
__device__ __forceinline__ unsigned next_ticket(uint32_t* sync, int lane, unsigned base)
{
    const unsigned t = atomicAdd(&sync[HF_SYNC_QUEUE], lane == 0 ? 1u : 0u);
    return __builtin_amdgcn_readfirstlane(t) + base;
}
// Tickets of a launch over items [0, n): wave w takes item w, then counter
// tickets.  When the items are no more than the waves, every wave takes at
// most its own item and no wave touches the counter: a wave would only learn
// there that the list is done, and those atomics all arrive together when the
// waves finish together and serialise at the counter.
__device__ __forceinline__ unsigned ticket_first(unsigned n, unsigned extra = 0)
{
    const unsigned w = wave_id();
    return (n <= total_waves(extra) && w >= n) ? n : w;   // otherwise w < waves < n
}
__device__ __forceinline__ unsigned ticket_next(uint32_t* sync, int lane, unsigned n, unsigned extra = 0)
{
    const unsigned nw = total_waves(extra);
    return n <= nw ? n : next_ticket(sync, lane, nw);
}

// What waves of one launch tell each other travels only through device-scope
// atomics (wave-speed maxima, fixed flags, the pending bitmap, the counters):
// writers update with atomic read-modify-writes, and
// readers of values that decide results read with coherent_read
// (hf_physics.h), an atomic read-modify-write that changes nothing.  The new
// states themselves are not read inside the launch.

// One item of the launch is complete.  This wave's atomics (its maxima and
// fixed flag) must be performed before the count that waiting waves poll:
// s_waitcnt vmcnt(0) waits until the memory system has acknowledged every
// vector memory operation this wave issued (atomics without return
// included), then the count is raised.
__device__ __forceinline__ void item_done(uint32_t* sync, int lane, unsigned n = 1)
{
    __builtin_amdgcn_s_waitcnt(0xF70);   // vmcnt(0), expcnt and lgkmcnt unconstrained
    __hip_atomic_fetch_add(&sync[HF_SYNC_DONE], lane == 0 ? n : 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Bounded wait until `target` items of the launch are complete (every item
// before position `target` of the queue: items are handed out in order and an
// item that waits never completes before the items it waits for).  The wait
// gives up after wait_ticks of the real-time counter (s_memrealtime, the
// clock HIP reports as hipDeviceAttributeWallClockRate), or at once when
// another wave has given up, and then returns false with the abort bit set:
// the caller leaves its item to the launch's last wave.  One load per poll
// (count and abort bit share a word); a load served late only delays the
// wait.
__device__ __forceinline__ bool wait_done(uint32_t* sync, unsigned target, unsigned long long wait_ticks)
{
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    for (;;) {
        const unsigned d = __builtin_amdgcn_readfirstlane(
            __hip_atomic_load(&sync[HF_SYNC_DONE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (d & HF_SYNC_ABORT_BIT) return false;
        if (d >= target) return true;
        if (__builtin_amdgcn_s_memrealtime() - t0 > wait_ticks) {
            __hip_atomic_fetch_or(&sync[HF_SYNC_DONE], HF_SYNC_ABORT_BIT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        __builtin_amdgcn_s_sleep(32);
    }
}

// A wave-reduced value as a wave-uniform (scalar) bit pattern.
__device__ __forceinline__ unsigned long long uniform_bits(double x)
{
    const unsigned long long b = dbits(x);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// Where a wave's maxima go: an array of slots and the wave's own slot of a
// block.  Device-scope atomics on one address take about 10 ns each, one
// after the other, so the waves of a launch are spread over a.ways slots on
// lines of their own (build_plan chooses how many).
struct MaxOut {
    unsigned long long* base;
    int way;
};
template <class R>
__device__ __forceinline__ MaxOut max_out(const HfStepArgs<R>& a, unsigned long long* base)
{
    return MaxOut{base, (int)(wave_id() & (unsigned)(a.ways - 1))};
}

// Per-wave maxima into the block's slots; every lane holds the reduced value.
// The value is passed as a scalar: the compiler then issues one atomic from
// one lane, instead of first reducing 64 lane values it cannot tell are equal
// (a 64-iteration scalar loop per atomic).
template <class R>
__device__ __forceinline__ void store_maxima(const HfStepArgs<R>& a, const MaxOut& out, int block, double mx, double my)
{
    const unsigned long long bx = uniform_bits(mx), by = uniform_bits(my);
    unsigned long long* p = out.base + HF_MAX_SLOT(block, out.way, a.ways, a.way_stride);
    atomicMax(p, bx);
    atomicMax(p + 1, by);
}

// x with its sign flipped where m (0 or the sign bit of a 32-bit word) says so.
__device__ __forceinline__ double flip_sign(double x, unsigned m)
{
    return __longlong_as_double(__double_as_longlong(x) ^ ((long long)((unsigned long long)m << 32)));
}
__device__ __forceinline__ float flip_sign(float x, unsigned m) { return __uint_as_float(__float_as_uint(x) ^ m); }

// A sweep's source of rows (T = false: lane l owns column x0 + l, lines are
// rows) or columns (T = true: lane l owns row y0 + l).  Ghost cells come from
// the filled ghost buffer; in a mirrored launch from the interior cell they
// mirror to, with the momentum normal to a reflective side negated (the fill
// of such a block puts the same values there: transmissive_boundary.cpp:25-104,
// reflective_boundary.cpp:25-120).  Corner ghosts, which no sweep uses, read
// cells inside the buffer.
template <class R, bool T>
struct Lines {
    const R* A;      // this lane's cell of line 0 (interior lines)
    const R* G;      // the same for ghost lines
    int64_t step, plane;
    int n, g;        // lines, ghost layers
    unsigned flip;   // this lane is mirrored at a reflective side
    unsigned lo, hi; // ghost lines below / above are mirrored at a reflective side
    bool mirrored;

    __device__ __forceinline__ Lines(const HfStepArgs<R>& a, const HfBlockDev& bd, int c)
    {
        mirrored = a.mirrored != 0;
        plane = bd.plane;
        g = bd.g;
        n = T ? bd.tx : bd.ty;
        step = T ? 1 : bd.pitch;
        const int m = T ? bd.ty : bd.tx;                    // lanes' extent
        const int64_t cs = T ? bd.pitch : 1;
        const bool below = c < g, ghost = below || c >= m - g;
        const int low = T ? 0 : 3, high = T ? 2 : 1;        // HF_BOTTOM/HF_TOP, HF_LEFT/HF_RIGHT
        const int llow = T ? 3 : 0, lhigh = T ? 1 : 2;
        flip = 0u;
        lo = hi = 0u;
        if (mirrored) {
            const int cm = !ghost ? c : below ? 2 * g - 1 - c : 2 * (m - g) - 1 - c;
            flip = (ghost && ((bd.reflect >> (below ? low : high)) & 1)) ? 0x80000000u : 0u;
            lo = ((bd.reflect >> llow) & 1) ? 0x80000000u : 0u;
            hi = ((bd.reflect >> lhigh) & 1) ? 0x80000000u : 0u;
            A = a.A + bd.off + cm * cs;
            G = A;
        } else {
            G = a.G + bd.off + c * cs;
            A = ghost ? G : a.A + bd.off + c * cs;
        }
    }
    // Requests line y into u: signs are applied by signed_line() with the
    // returned mask, apart, so that nothing waits for the load here.
    __device__ __forceinline__ unsigned operator()(int y, R u[4]) const
    {
        const bool below = y < g, ghost = below || y >= n - g;   // wave-uniform
        const int ym = !(ghost && mirrored) ? y : below ? 2 * g - 1 - y : 2 * (n - g) - 1 - y;
        load_cell<R>((ghost ? G : A) + ym * step, plane, u);
        return below ? lo : ghost ? hi : 0u;
    }
    __device__ __forceinline__ void signed_line(R u[4], unsigned f) const
    {
        constexpr int L = T ? 2 : 1, N = T ? 1 : 2;   // momenta normal to the lanes' and the lines' sides
        u[L] = flip_sign(u[L], flip);
        u[N] = flip_sign(u[N], f);
    }
};

// ---------------------------------------------------------- MUSCL-Hancock --
// The step dt and the half steps dt_pred / (2 dx), dt_pred / (2 dy) (half_dt_dx,
// muscl_hancock.cpp:248) of an item of block bd.
template <class Dts>
__device__ __forceinline__ void half_steps(const HfBlockDev& bd, Dts&& dts, double& dt_step, double& hx, double& hy)
{
    double dt_pred;
    dts(dt_step, dt_pred);
    hx = (0.5 * dt_pred) / bd.dx;
    hy = (0.5 * dt_pred) / bd.dy;
}

// Rows of an item in range (q64 in hf_physics.h), from the first on: returns
// the number of rows done, it.rows unless a lane left the range.  The caller
// finishes with the general rows.
// Per row: the new row's differences to the one before it serve the y slopes
// of this row and, kept, of the next; the x slopes take theirs from the right
// neighbour, and the left one's by a lane shift.
// FP64 VALU issue bounds it, with two waves per SIMD: 8192^2 Van Leer runs at
// 27.5 Gcell-updates/s, 21.5 with the general rows.
template <class M, int LIM, class Dts>
__device__ __forceinline__ int muscl_rows_q64(const HfStepArgs<double>& a, const HfItem it, const HfBlockDev& bd,
                                              const int lane, Dts&& dts, double& dt_step, double& hx, double& hy,
                                              double& mx, double& my)
{
    const double gam = a.gamma, g1 = a.gamma - 1.0;
    const double ig1 = 1.0 / g1;
    const q64::Limits lim;
    const int xraw = it.x0 + lane;
    const bool valid = xraw < bd.tx;
    const int xc = valid ? xraw : bd.tx - 1;
    const Lines<double, false> ROW(a, bd, xc);
    const int pitch = bd.pitch, ty = bd.ty;
    const int64_t plane = bd.plane;
    const bool out = valid && lane >= 2 && lane < 62 && xraw >= 2 && xraw < bd.tx - 2;
    // lanes that write, whose x faces those use, and that those are reconstructed from
    const q64::mask m0 = __ballot(out), m1 = m0 | m0 << 1 | m0 >> 1, m2 = m1 | m1 << 1 | m1 >> 1;
    const double rdx = 1.0 / bd.dx, rdy = 1.0 / bd.dy;

    const int y0 = it.y0;
    double uc[4], up[4], un[4], dl[4], cl[4], Gs[4], Tc[4];
    q64::mask bad = 0, bc, bp, bn;   // rows y, y+1, y+2 out of range
    {
        double um[4], dr[4], cr[4], lo[4], hi[4];
        const unsigned fm = ROW(y0 - 2, um), fc = ROW(y0 - 1, uc), fp = ROW(y0, up), fn = ROW(y0 + 1, un);
        half_steps(bd, dts, dt_step, hx, hy);   // behind the loads: its own chain of loads overlaps theirs
        if (!(q64::constants_in_range(gam, g1) && q64::half_step_in_range(hx) && q64::half_step_in_range(hy))) return 0;
        ROW.signed_line(um, fm);
        ROW.signed_line(uc, fc);
        ROW.signed_line(up, fp);
        ROW.signed_line(un, fn);
        bad = q64::out_of_range(um, lim) | q64::out_of_range(uc, lim);
        bc = q64::out_of_range(up, lim);
        bp = q64::out_of_range(un, lim);
        if ((bad | bc | bp) & m0) return 0;   // before arithmetic that would be done twice
        q64::differences(um, uc, dl, cl, lim);
        q64::differences(uc, up, dr, cr, lim);
        q64::reconstruct<LIM, false>(uc, dl, dr, cl, cr, hy, g1, ig1, lo, hi, bad, lim);     // cell y0-1
        const q64::State sl = q64::make_state(hi, gam, g1, ig1, bad, lim);
        q64::differences(up, un, dl, cl, lim);
        q64::reconstruct<LIM, false>(up, dr, dl, cr, cl, hy, g1, ig1, lo, Tc, bad, lim);     // cell y0
        const q64::State sr = q64::make_state(lo, gam, g1, ig1, bad, lim);
        q64::hllc<false>(sl, sr, Gs, bad, lim);
        if ((bad | bc | bp) & m0) return 0;
    }
    for (int k = 0; k < 4; k++) { uc[k] = up[k]; up[k] = un[k]; }
    unsigned fn = ROW(y0 + 2, un);

    double* Ob = a.O + bd.off;
    for (int r = 0; r < it.rows; r++) {
        const int y = y0 + r;
        double nn[4];
        ROW.signed_line(un, fn);
        fn = ROW(y + 3 < ty ? y + 3 : ty - 1, nn);     // next iteration's U(y+2)
        bn = q64::out_of_range(un, lim);

        // y direction: reconstruct cell y+1, flux through face y+1/2
        q64::mask by = 0, bx = 0;
        double dn[4], cn[4], Bn[4], Tn[4], Gn[4];
        q64::differences(up, un, dn, cn, lim);
        q64::reconstruct<LIM, false>(up, dl, dn, cl, cn, hy, g1, ig1, Bn, Tn, by, lim);
        {
            const q64::State sl = q64::make_state(Tc, gam, g1, ig1, by, lim);
            const q64::State sr = q64::make_state(Bn, gam, g1, ig1, by, lim);
            q64::hllc<false>(sl, sr, Gn, by, lim);
        }

        // x direction: reconstruct cell (x, y) from lane neighbours
        double ur[4], xl[4], xr[4], kl[4], kr[4], Lf[4], Rf[4], Rl[4], Fw[4], Fe[4];
        for (int k = 0; k < 4; k++) ur[k] = shfl_dn1(uc[k]);
        q64::differences(uc, ur, xr, kr, lim);
        for (int k = 0; k < 4; k++) { xl[k] = shfl_up1(xr[k]); kl[k] = shfl_up1(kr[k]); }
        q64::reconstruct<LIM, true>(uc, xl, xr, kl, kr, hx, g1, ig1, Lf, Rf, bx, lim);
        for (int k = 0; k < 4; k++) Rl[k] = shfl_up1(Rf[k]);
        {
            const q64::State sl = q64::make_state(Rl, gam, g1, ig1, bx, lim);
            const q64::State sr = q64::make_state(Lf, gam, g1, ig1, bx, lim);
            q64::hllc<true>(sl, sr, Fw, bx, lim);          // face x-1/2
        }
        for (int k = 0; k < 4; k++) Fe[k] = shfl_dn1(Fw[k]);   // face x+1/2

        double Ln[4], Un[4], dx_, dy_;
        update_cell<M>(rdx, rdy, dt_step, Fw, Fe, Gs, Gn, uc, Ln, Un);
        q64::wave_speeds(Un, gam, g1, dx_, dy_, by, lim);
        if (((by | bp | bn) & m0) | (bx & m1) | (bc & m2)) return r;
        if (out) {
            double* o = Ob + (int64_t)y * pitch + xraw;
            for (int k = 0; k < 4; k++) o[k * plane] = Un[k];
            mx = dmax_nan(mx, dx_);
            my = dmax_nan(my, dy_);
        }
        bc = bp;
        bp = bn;
        for (int k = 0; k < 4; k++) {
            Gs[k] = Gn[k]; Tc[k] = Tn[k]; uc[k] = up[k]; up[k] = un[k]; un[k] = nn[k];
            dl[k] = dn[k]; cl[k] = cn[k];
        }
    }
    return it.rows;
}

// MUSCLHancockScheme::operator() (scheme/muscl_hancock/muscl_hancock.cpp:41-55)
// fused with ForwardEulerODESolver (scheme/ode/forward_euler/forward_euler.cpp:25-30).
// Output columns per wave: 60 (lanes 2..61); lanes 0,1,62,63 are halo.
template <class M, int LIM, bool RESID, bool QUICK, class Dts>
__device__ __forceinline__ void muscl_item(const HfStepArgs<typename M::R>& a, const HfItem it, const int lane,
                                           Dts&& dts, const MaxOut& imax_out)
{
    typedef typename M::R R;

    const HfBlockDev bd = a.blocks[it.block];
    const int xraw = it.x0 + lane;
    const bool valid = xraw < bd.tx;
    const int xc = valid ? xraw : bd.tx - 1;
    const Lines<R, false> ROW(a, bd, xc);
    const int pitch = bd.pitch, ty = bd.ty;
    const int64_t plane = bd.plane;
    const bool out = valid && lane >= 2 && lane < 62 && xraw >= 2 && xraw < bd.tx - 2;

    const R rdx = R(1.0 / bd.dx);                  // one_dx, muscl_hancock.cpp:352
    const R rdy = R(1.0 / bd.dy);
    double dt_step, hx_, hy_;
    const R gam = R(a.gamma), g1 = R(a.gamma - 1.0);

    double mx = 0.0, my = 0.0;
    int done = 0;
    constexpr bool IN_RANGE = QUICK && !RESID && !M::fast;
    if constexpr (IN_RANGE) done = muscl_rows_q64<M, LIM>(a, it, bd, lane, dts, dt_step, hx_, hy_, mx, my);
    if (done < it.rows) {
    const int y0 = it.y0 + done, rows = it.rows - done;
    R um[4], uc[4], up[4], un[4];
    const unsigned fm = ROW(y0 - 2, um), fc = ROW(y0 - 1, uc), fp = ROW(y0, up);
    unsigned fn = ROW(y0 + 1, un);
    if (!IN_RANGE) half_steps(bd, dts, dt_step, hx_, hy_);
    ROW.signed_line(um, fm);
    ROW.signed_line(uc, fc);
    ROW.signed_line(up, fp);
    ROW.signed_line(un, fn);
    const R hx = R(hx_), hy = R(hy_), dtR = R(dt_step);

    // warm-up: T' of cell y0-1, (B', T') of cell y0, flux through face y0-1/2
    R G0[4], G1[4], T0[4], T1[4];
    {
        R lo[4], hi[4];
        reconstruct<M, LIM, false>(um, uc, up, hy, g1, lo, hi);   // cell y0-1
        R lo2[4];
        reconstruct<M, LIM, false>(uc, up, un, hy, g1, lo2, T0);  // cell y0
        const State<R> sl = make_state<M>(hi, gam, g1);
        const State<R> sr = make_state<M>(lo2, gam, g1);
        hllc<M, false>(sl, sr, G0);
    }
    // The window of rows y, y+1, y+2 and the one loaded an iteration ahead so
    // that HBM latency overlaps the row's arithmetic.  In FP32, bound by VALU
    // issue, its four arrays change their parts from row to row by name, with the
    // row's code four times in the loop: moving them took 27 more instructions.
    // A Van Leer row went from 498 instructions to 409 with this, with shared
    // differences and with the median in slope(): 8192^2 860 -> 800 us a step,
    // 4096^2 250 -> 231, 1024^2 26.3 -> 25.8, 512^2 14.8 -> 13.5.  Four waves per
    // SIMD (9 registers spilled) took 768, 256, 28.3 and 13.8.
    R W0[4], W1[4], W2[4], W3[4], D0[4], D1[4], C0[4], C1[4];   // D, C: FP32, U(y+1) - U(y), raw and clamped
    for (int k = 0; k < 4; k++) { W0[k] = up[k]; W1[k] = un[k]; }
    fn = ROW(y0 + 2, W2);
    if constexpr (M::fast) f32::differences(W0, W1, D0, C0);

    R* Ob = RESID ? a.O : a.O + bd.off;
    auto step = [&](int r, R (&uc)[4], R (&up)[4], R (&un)[4], R (&nn)[4], R (&dl)[4], R (&cl)[4], R (&dn)[4],
                    R (&cn)[4], R (&Gs)[4], R (&Gn)[4], R (&Tc)[4], R (&Tn)[4]) {
        const int y = y0 + r;
        ROW.signed_line(un, fn);
        fn = ROW(y + 3 < ty ? y + 3 : ty - 1, nn);     // next iteration's U(y+2)

        // y direction: reconstruct cell y+1, flux through face y+1/2
        R Bn[4];
        if constexpr (M::fast) {
            f32::differences(up, un, dn, cn);
            f32::reconstruct<LIM, false>(up, dl, dn, cl, cn, hy, g1, Bn, Tn);
        } else {
            reconstruct<M, LIM, false>(uc, up, un, hy, g1, Bn, Tn);
        }
        {
            const State<R> sl = make_state<M>(Tc, gam, g1);
            const State<R> sr = make_state<M>(Bn, gam, g1);
            hllc<M, false>(sl, sr, Gn);
        }

        // x direction: reconstruct cell (x, y) from lane neighbours
        R ur[4], Lf[4], Rf[4], Rl[4], Fw[4], Fe[4];
        for (int k = 0; k < 4; k++) ur[k] = shfl_dn1(uc[k]);
        if constexpr (M::fast) {
            R xl[4], xr[4], kl[4], kr[4];
            f32::differences(uc, ur, xr, kr);
            for (int k = 0; k < 4; k++) { xl[k] = shfl_up1(xr[k]); kl[k] = shfl_up1(kr[k]); }
            f32::reconstruct<LIM, true>(uc, xl, xr, kl, kr, hx, g1, Lf, Rf);
        } else {
            R ul[4];
            for (int k = 0; k < 4; k++) ul[k] = shfl_up1(uc[k]);
            reconstruct<M, LIM, true>(ul, uc, ur, hx, g1, Lf, Rf);
        }
        for (int k = 0; k < 4; k++) Rl[k] = shfl_up1(Rf[k]);
        {
            const State<R> sl = make_state<M>(Rl, gam, g1);
            const State<R> sr = make_state<M>(Lf, gam, g1);
            hllc<M, true>(sl, sr, Fw);          // face x-1/2
        }
        for (int k = 0; k < 4; k++) Fe[k] = shfl_dn1(Fw[k]);   // face x+1/2

        // calculate_spatial_update (muscl_hancock.cpp:364-371) and (dt*L)+U
        R Ln[4], Un[4];
        update_cell<M>(rdx, rdy, dtR, Fw, Fe, Gs, Gn, uc, Ln, Un);
        if (out) {
            R* o = Ob + (int64_t)y * pitch;
            for (int k = 0; k < 4; k++) (o + k * plane)[(uint32_t)xraw] = RESID ? Ln[k] : Un[k];
            if (!RESID) {
                double dx_, dy_;
                wave_speeds<M>(Un[0], Un[1], Un[2], Un[3], gam, g1, dx_, dy_);
                mx = dmax_nan(mx, dx_);
                my = dmax_nan(my, dy_);
            }
        }
    };
    for (int r = 0;;) {
        step(r, W0, W1, W2, W3, D0, C0, D1, C1, G0, G1, T0, T1);
        if (++r >= rows) break;
        if constexpr (M::fast) {
            step(r, W1, W2, W3, W0, D1, C1, D0, C0, G1, G0, T1, T0);
            if (++r >= rows) break;
            step(r, W2, W3, W0, W1, D0, C0, D1, C1, G0, G1, T0, T1);
            if (++r >= rows) break;
            step(r, W3, W0, W1, W2, D1, C1, D0, C0, G1, G0, T1, T0);
            if (++r >= rows) break;
        } else {
            for (int k = 0; k < 4; k++) {
                G0[k] = G1[k]; T0[k] = T1[k]; W0[k] = W1[k]; W1[k] = W2[k]; W2[k] = W3[k];
            }
        }
    }
    }
    if (!RESID) store_maxima(a, imax_out, it.block, wave_max(mx), wave_max(my));
}

// The same update for a narrow column band at a block's right edge, with the
// roles of x and y exchanged: lane l owns padded row it.y0 + l and the wave
// walks along the band's columns.  A block whose width leaves a last column
// strip with only a few output columns (1024 = 17 x 60 + 4) would otherwise
// spend a whole wave per row on them.  Every face state, flux and update is
// the same function of the same operands as in muscl_item, in the same order,
// so the results are identical.  Item encoding: rows = -(cols + 256 * nrows),
// x0 = first output column (padded), y0 = padded row of lane 0; lanes 2..61
// write, up to nrows of them.
__device__ __forceinline__ bool item_transposed(const HfItem& it) { return it.rows < 0; }

// Columns of a transposed item in range, as muscl_rows_q64.
template <class M, int LIM, class Dts>
__device__ __forceinline__ int muscl_cols_q64(const HfStepArgs<double>& a, const HfItem it, const HfBlockDev& bd,
                                              const int lane, Dts&& dts, double& dt_step, double& hx, double& hy,
                                              double& mx, double& my)
{
    const double gam = a.gamma, g1 = a.gamma - 1.0;
    const double ig1 = 1.0 / g1;
    const q64::Limits lim;
    const int code = -it.rows;
    const int cols = code & 255, nrows = code >> 8;
    const int yraw = it.y0 + lane;
    const bool valid = yraw < bd.ty;
    const int yc = valid ? yraw : bd.ty - 1;
    const Lines<double, true> COL(a, bd, yc);
    const int pitch = bd.pitch, tx = bd.tx;
    const int64_t plane = bd.plane;
    const bool out = valid && lane >= 2 && lane < 62 && lane < 2 + nrows && yraw >= 2 && yraw < bd.ty - 2;
    const q64::mask m0 = __ballot(out), m1 = m0 | m0 << 1 | m0 >> 1, m2 = m1 | m1 << 1 | m1 >> 1;
    const double rdx = 1.0 / bd.dx, rdy = 1.0 / bd.dy;

    const int x0 = it.x0;
    double uc[4], up[4], un[4], dl[4], cl[4], Fw[4], Rc[4];
    q64::mask bad = 0, bc, bp, bn;   // columns x, x+1, x+2 out of range
    {
        double um[4], dr[4], cr[4], lo[4], hi[4];
        const unsigned fm = COL(x0 - 2, um), fc = COL(x0 - 1, uc), fp = COL(x0, up), fn = COL(x0 + 1, un);
        half_steps(bd, dts, dt_step, hx, hy);   // behind the loads: its own chain of loads overlaps theirs
        if (!(q64::constants_in_range(gam, g1) && q64::half_step_in_range(hx) && q64::half_step_in_range(hy))) return 0;
        COL.signed_line(um, fm);
        COL.signed_line(uc, fc);
        COL.signed_line(up, fp);
        COL.signed_line(un, fn);
        bad = q64::out_of_range(um, lim) | q64::out_of_range(uc, lim);
        bc = q64::out_of_range(up, lim);
        bp = q64::out_of_range(un, lim);
        if ((bad | bc | bp) & m0) return 0;   // before arithmetic that would be done twice
        q64::differences(um, uc, dl, cl, lim);
        q64::differences(uc, up, dr, cr, lim);
        q64::reconstruct<LIM, true>(uc, dl, dr, cl, cr, hx, g1, ig1, lo, hi, bad, lim);      // column x0-1
        const q64::State sl = q64::make_state(hi, gam, g1, ig1, bad, lim);
        q64::differences(up, un, dl, cl, lim);
        q64::reconstruct<LIM, true>(up, dr, dl, cr, cl, hx, g1, ig1, lo, Rc, bad, lim);      // column x0
        const q64::State sr = q64::make_state(lo, gam, g1, ig1, bad, lim);
        q64::hllc<true>(sl, sr, Fw, bad, lim);
        if ((bad | bc | bp) & m0) return 0;
    }
    for (int k = 0; k < 4; k++) { uc[k] = up[k]; up[k] = un[k]; }
    unsigned fn = COL(x0 + 2, un);

    double* Ob = a.O + bd.off;
    for (int c = 0; c < cols; c++) {
        const int x = x0 + c;
        double nn[4];
        COL.signed_line(un, fn);
        fn = COL(x + 3 < tx ? x + 3 : tx - 1, nn);     // next iteration's U(x+2)
        bn = q64::out_of_range(un, lim);

        // x direction: reconstruct column x+1, flux through face x+1/2
        q64::mask by = 0, bx = 0;
        double dn[4], cn[4], Ln[4], Rn[4], Fe[4];
        q64::differences(up, un, dn, cn, lim);
        q64::reconstruct<LIM, true>(up, dl, dn, cl, cn, hx, g1, ig1, Ln, Rn, bx, lim);
        {
            const q64::State sl = q64::make_state(Rc, gam, g1, ig1, bx, lim);
            const q64::State sr = q64::make_state(Ln, gam, g1, ig1, bx, lim);
            q64::hllc<true>(sl, sr, Fe, bx, lim);
        }

        // y direction: reconstruct cell (x, y) from lane neighbours
        double ut[4], xl[4], xr[4], kl[4], kr[4], Bf[4], Tf[4], Tl[4], Gs[4], Gn[4];
        for (int k = 0; k < 4; k++) ut[k] = shfl_dn1(uc[k]);
        q64::differences(uc, ut, xr, kr, lim);
        for (int k = 0; k < 4; k++) { xl[k] = shfl_up1(xr[k]); kl[k] = shfl_up1(kr[k]); }
        q64::reconstruct<LIM, false>(uc, xl, xr, kl, kr, hy, g1, ig1, Bf, Tf, by, lim);
        for (int k = 0; k < 4; k++) Tl[k] = shfl_up1(Tf[k]);
        {
            const q64::State sl = q64::make_state(Tl, gam, g1, ig1, by, lim);
            const q64::State sr = q64::make_state(Bf, gam, g1, ig1, by, lim);
            q64::hllc<false>(sl, sr, Gs, by, lim);         // face y-1/2
        }
        for (int k = 0; k < 4; k++) Gn[k] = shfl_dn1(Gs[k]);   // face y+1/2

        double Lu[4], Un[4], dx_, dy_;
        update_cell<M>(rdx, rdy, dt_step, Fw, Fe, Gs, Gn, uc, Lu, Un);
        q64::wave_speeds(Un, gam, g1, dx_, dy_, bx, lim);
        if (((bx | bp | bn) & m0) | (by & m1) | (bc & m2)) return c;
        if (out) {
            double* o = Ob + (int64_t)yraw * pitch + x;
            for (int k = 0; k < 4; k++) o[k * plane] = Un[k];
            mx = dmax_nan(mx, dx_);
            my = dmax_nan(my, dy_);
        }
        bc = bp;
        bp = bn;
        for (int k = 0; k < 4; k++) {
            Fw[k] = Fe[k]; Rc[k] = Rn[k]; uc[k] = up[k]; up[k] = un[k]; un[k] = nn[k];
            dl[k] = dn[k]; cl[k] = cn[k];
        }
    }
    return cols;
}

template <class M, int LIM, bool RESID, bool QUICK, class Dts>
__device__ __forceinline__ void muscl_item_t(const HfStepArgs<typename M::R>& a, const HfItem it, const int lane,
                                             Dts&& dts, const MaxOut& imax_out)
{
    typedef typename M::R R;

    const HfBlockDev bd = a.blocks[it.block];
    const int code = -it.rows;
    const int cols = code & 255, nrows = code >> 8;
    const int yraw = it.y0 + lane;
    const bool valid = yraw < bd.ty;
    const int yc = valid ? yraw : bd.ty - 1;
    const Lines<R, true> COL(a, bd, yc);
    const int pitch = bd.pitch, tx = bd.tx;
    const int64_t plane = bd.plane;
    const bool out = valid && lane >= 2 && lane < 62 && lane < 2 + nrows && yraw >= 2 && yraw < bd.ty - 2;

    const R rdx = R(1.0 / bd.dx);                  // one_dx, muscl_hancock.cpp:352
    const R rdy = R(1.0 / bd.dy);
    double dt_step, hx_, hy_;
    const R gam = R(a.gamma), g1 = R(a.gamma - 1.0);

    double mx = 0.0, my = 0.0;
    int done = 0;
    constexpr bool IN_RANGE = QUICK && !RESID && !M::fast;
    if constexpr (IN_RANGE)
        done = muscl_cols_q64<M, LIM>(a, it, bd, lane, dts, dt_step, hx_, hy_, mx, my);
    if (done < cols) {
    const int x0 = it.x0 + done, left = cols - done;
    R um[4], uc[4], up[4], un[4];
    const unsigned fm = COL(x0 - 2, um), fc = COL(x0 - 1, uc), fp = COL(x0, up);
    unsigned fn = COL(x0 + 1, un);
    if (!IN_RANGE) half_steps(bd, dts, dt_step, hx_, hy_);
    COL.signed_line(um, fm);
    COL.signed_line(uc, fc);
    COL.signed_line(up, fp);
    COL.signed_line(un, fn);
    const R hx = R(hx_), hy = R(hy_), dtR = R(dt_step);

    // warm-up: R' of column x0-1, (L', R') of column x0, flux through face x0-1/2
    R Fw[4], Rc[4];
    {
        R lo[4], hi[4];
        reconstruct<M, LIM, true>(um, uc, up, hx, g1, lo, hi);    // column x0-1
        R lo2[4];
        reconstruct<M, LIM, true>(uc, up, un, hx, g1, lo2, Rc);   // column x0
        const State<R> sl = make_state<M>(hi, gam, g1);
        const State<R> sr = make_state<M>(lo2, gam, g1);
        hllc<M, true>(sl, sr, Fw);
    }
    for (int k = 0; k < 4; k++) { uc[k] = up[k]; up[k] = un[k]; }
    fn = COL(x0 + 2, un);

    R* Ob = RESID ? a.O : a.O + bd.off;
    for (int c = 0; c < left; c++) {
        const int x = x0 + c;
        R nn[4];
        COL.signed_line(un, fn);
        fn = COL(x + 3 < tx ? x + 3 : tx - 1, nn);     // next iteration's U(x+2)

        // x direction: reconstruct column x+1, flux through face x+1/2
        R Ln[4], Rn[4], Fe[4];
        reconstruct<M, LIM, true>(uc, up, un, hx, g1, Ln, Rn);
        {
            const State<R> sl = make_state<M>(Rc, gam, g1);
            const State<R> sr = make_state<M>(Ln, gam, g1);
            hllc<M, true>(sl, sr, Fe);
        }

        // y direction: reconstruct cell (x, y) from lane neighbours
        R ub[4], ut[4], Bf[4], Tf[4], Tl[4], Gs[4], Gn[4];
        for (int k = 0; k < 4; k++) { ub[k] = shfl_up1(uc[k]); ut[k] = shfl_dn1(uc[k]); }
        reconstruct<M, LIM, false>(ub, uc, ut, hy, g1, Bf, Tf);
        for (int k = 0; k < 4; k++) Tl[k] = shfl_up1(Tf[k]);
        {
            const State<R> sl = make_state<M>(Tl, gam, g1);
            const State<R> sr = make_state<M>(Bf, gam, g1);
            hllc<M, false>(sl, sr, Gs);         // face y-1/2
        }
        for (int k = 0; k < 4; k++) Gn[k] = shfl_dn1(Gs[k]);   // face y+1/2

        // calculate_spatial_update (muscl_hancock.cpp:364-371) and (dt*L)+U
        R Lu[4], Un[4];
        update_cell<M>(rdx, rdy, dtR, Fw, Fe, Gs, Gn, uc, Lu, Un);
        if (out) {
            R* o = Ob + (int64_t)yraw * pitch + x;
            for (int k = 0; k < 4; k++) o[k * plane] = RESID ? Lu[k] : Un[k];
            if (!RESID) {
                double dx_, dy_;
                wave_speeds<M>(Un[0], Un[1], Un[2], Un[3], gam, g1, dx_, dy_);
                mx = dmax_nan(mx, dx_);
                my = dmax_nan(my, dy_);
            }
        }
        for (int k = 0; k < 4; k++) { Fw[k] = Fe[k]; Rc[k] = Rn[k]; uc[k] = up[k]; up[k] = un[k]; un[k] = nn[k]; }
    }
    }
    if (!RESID) store_maxima(a, imax_out, it.block, wave_max(mx), wave_max(my));
}

// The guess launch's plan of problem p (plan_scan with the main list's
// maxima): its first block to fix, the guess minimum m and the speculative
// minimum O; t: the terms of the first 64 blocks, for a plan_scan that follows.
template <class R>
__device__ __forceinline__ int guess_plan(const HfStepArgs<R>& a, int p, const HfProbDev& pr, double& O, double& m,
                                          long long& kstep, PlanTerms& t)
{
    kstep = (long long)a.calls[p] - pr.cps + 1;
    t = plan_terms<R>(a, pr, a.nblocks);
    double o = smin(1e16, t.o);
    const int end = pr.first + pr.nb;
    for (int c = pr.first + 64 + (int)(threadIdx.x & 63); c < end; c += 64) o = smin(o, term_old(a, c));
    O = wave_min(o);
    m = 0.0;
    return plan_scan<R, PRE_MAIN>(a, pr, a.nblocks, kstep, O, t, m, false);
}
template <class R>
__device__ __forceinline__ int guess_plan(const HfStepArgs<R>& a, int p, const HfProbDev& pr, double& O, double& m,
                                          long long& kstep)
{
    PlanTerms t;
    return guess_plan<R>(a, p, pr, O, m, kstep, t);
}

// What a wave of the check launch knows of a block (verdict_on), and of its
// problem: the guess minimum, which the launch does not change.  A wave that
// goes through the rounds takes them from here instead of planning again for
// every round and item: the check launch of a step that recomputes blocks of the
// 8 x 97^2 channel took 185 us with that, 160 without.
struct Verdict {
    int block = -1, problem = -1;
    bool need = false;
    double mg = 0.0, step = 0.0, pred = 0.0;
    long long kstep = 0, kpred = 0;
};
template <class R>
__device__ __forceinline__ void verdict_on(const HfStepArgs<R>& a, int p, const HfProbDev& pr, int lb, Verdict& v)
{
    if (p != v.problem) {
        double O;
        guess_plan<R>(a, p, pr, O, v.mg, v.kstep);
        v.problem = p;
    }
    v.block = pr.first + lb;
    v.need = check_verdict<R>(a, p, pr, a.nblocks, lb, v.mg, v.step, v.pred, v.kstep, v.kpred);
}

// Check-launch rounds from round l on, while none of their blocks needs
// computing: round l holds the l-th block of every problem with more than l
// blocks, and its verdicts need the blocks before it final, which holds while
// every earlier round has been completed.  The queue counter jumps past each
// round passed over (its unissued items are counted complete).  Returns the
// first round to compute, or nrounds + 1; v keeps the last verdict.
template <class R>
__device__ int first_busy_round(const HfStepArgs<R>& a, int l, int lane, unsigned base, Verdict& v)
{
    for (; l <= a.nrounds; l++) {
        bool need = false;
        for (int p = 0; p < a.nprob; p++) {
            const HfProbDev pr = a.probs[p];
            if (pr.nb <= l) continue;
            verdict_on<R>(a, p, pr, l, v);
            need = v.need || need;
        }
        if (need) return l;
        const unsigned end = (unsigned)a.rounds[l + 1] - base;
        const unsigned old = __builtin_amdgcn_readfirstlane(atomicMax(&a.sync[HF_SYNC_QUEUE], end));
        if (old < end) item_done(a.sync, lane, end - old);
    }
    return a.nrounds + 1;
}

// Which fix-up round an item position belongs to (rounds are few).
template <class R>
__device__ __forceinline__ int round_of(const HfStepArgs<R>& a, unsigned idx)
{
    int l = 1;
    while (l < a.nrounds && idx >= (unsigned)a.rounds[l + 1]) l++;
    return l;
}

// dts(step, pred) gives the item's step and predictor dt; it is called once,
// after the item's first lines are requested.
template <class M, int LIM, bool RESID, bool QUICK = true, class Dts>
__device__ __forceinline__ void muscl_go(const HfStepArgs<typename M::R>& a, const HfItem& it, int lane, Dts&& dts,
                                         const MaxOut& imax_out)
{
    if (!RESID && item_transposed(it))
        muscl_item_t<M, LIM, RESID, QUICK>(a, it, lane, dts, imax_out);
    else
        muscl_item<M, LIM, RESID, QUICK>(a, it, lane, dts, imax_out);
}

template <class R>
__device__ __forceinline__ void record_dts(const HfStepArgs<R>& a, const HfItem& it, const HfBlockDev& bd, bool step,
                                           double dt_step, double dt_pred, long long kstep, long long kpred)
{
    if (bd.problem == 0 && it.x0 == 0 && it.y0 == bd.g) {   // same value from every lane
        const long long hs = kstep - a.hist_base, hp = kpred - a.hist_base;
        if (step && bd.lb == 0 && hs >= 1 && hs <= a.hist_cap) a.hist[hs - 1] = dt_step;
        if (hp >= 1 && hp <= a.hist_cap) a.hist[hp - 1] = dt_pred;
    }
}

// MUSCL-Hancock step with the reference-compatible dt (muscl_hancock.cpp:246
// with the sequential block loop of simulation.cpp:106-110: block l's
// predictor dt sees blocks 0..l-1 of its problem at U^{n+1}) in three
// persistent launches, each writing a block at most once (the XCDs' L2 caches
// are written back in no fixed order, so two writers of one cache line in one
// launch could leave either value):
//  1. main (k_muscl): every block except those marked skip[b] (the previous
//     step's verdict that the speculation fails), with the speculative
//     predictor dt (every block at U^n).  No block waits for another.
//  2. guess (k_muscl_guess): from the main list's maxima, each problem's
//     first wrong block L and, for every block l >= L, the exact dt of block
//     L scaled to l -- exact for l as long as blocks L..l-1 do not set a new
//     minimum.  Every block whose dt differs from its speculative one (or
//     that was skipped) is computed with it.  No waits.
//  3. check (k_muscl_check): from the final maxima, the first block whose dt
//     so far is not the exact one; normally none, and the launch returns at
//     once.  Otherwise rounds follow from that block on: round l holds block
//     l of every problem and waits (bounded) until every earlier round is
//     complete, then recomputes the blocks whose dt is still wrong.
// Items [0, nmain) form the main list, [nmain, nitems) the rounds: round l
// lists the l-th block of every problem (the guess and check launches take
// them in that order).  Without a CFL dt (use_fixed) or in uniform mode the
// main launch is the whole step.
// Exclusive prefix sum over the wave's lanes; total: the sum over all lanes.
__device__ __forceinline__ unsigned lane_prefix(unsigned x, unsigned& total)
{
    const int lane = threadIdx.x & 63;
    unsigned v = x;
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned o = __shfl_up(v, d, 64);
        if (lane >= d) v += o;
    }
    total = __builtin_amdgcn_readlane(v, 63);
    return v - x;
}

// A ticket of a launch that takes only some of its item ranges: the ranges
// are visited 64 at a time (lane <-> range), each lane holding its range's
// first item, its count (0: not taken) and the items of the taken ranges
// before it in the chunk.  Tickets count taken items only, so no ticket is
// spent on an item that is not computed; a wave's tickets only grow, so its
// cursor only moves forward.
struct RangeCursor {
    int c0;            // first range of the current chunk
    unsigned base;     // taken items before the chunk
    unsigned total;    // taken items in the chunk
    int first;         // this lane's range: first item
    unsigned cnt, pre; // this lane's range: taken items, taken items before it in the chunk
};

// Item position of ticket t in the chunk that holds it: the lane whose range
// covers it, and the item.
__device__ __forceinline__ unsigned cursor_item(const RangeCursor& cur, unsigned t, int& lane_of)
{
    const unsigned r = t - cur.base;
    const unsigned long long bal = __ballot(cur.cnt > 0u && r >= cur.pre && r < cur.pre + cur.cnt);
    if (!bal) return 0xffffffffu;   // not reached: the chunk's ranges cover [base, base + total)
    lane_of = __builtin_ctzll(bal);
    const unsigned pre = __builtin_amdgcn_readlane(cur.pre, lane_of);
    const int first = __builtin_amdgcn_readlane(cur.first, lane_of);
    return (unsigned)first + (r - pre);
}

// Main list with skipped blocks: ranges are the (phase, block) segments in
// list order, a segment taken unless its block is skipped.
template <class R>
__device__ __forceinline__ void main_chunk(const HfStepArgs<R>& a, RangeCursor& cur, int c0)
{
    const int k = c0 + (int)(threadIdx.x & 63);
    const int nseg = 3 * a.nblocks;
    cur.c0 = c0;
    cur.first = 0;
    cur.cnt = 0u;
    if (k < nseg && !a.skip[k % a.nblocks]) {
        cur.first = a.segs[2 * k];
        cur.cnt = (unsigned)a.segs[2 * k + 1];
    }
    cur.pre = lane_prefix(cur.cnt, cur.total);
}

template <class M, int LIM, bool RESID>
__device__ __forceinline__ void main_item(const HfStepArgs<typename M::R>& a, unsigned idx, int lane, int& cached,
                                          double& c_step, double& c_pred, long long& c_kstep, long long& c_kpred)
{
    typedef typename M::R R;
    const HfItem it = a.items[a.item0 + idx];
    if (!a.use_fixed && !a.mirrored && a.skip[it.block]) return;   // left to the guess launch
    auto dts = [&](double& step, double& pred) {
        if (a.use_fixed) {
            step = a.fixed_step;
            pred = a.fixed_pred;
            return;
        }
        const HfBlockDev bd = a.blocks[it.block];
        if (it.block != cached) {
            cached = it.block;
            step_dts<R>(a, bd, true, c_step, c_pred, c_kstep, c_kpred);
        }
        record_dts<R>(a, it, bd, true, c_step, c_pred, c_kstep, c_kpred);
        step = c_step;
        pred = c_pred;
    };
    muscl_go<M, LIM, RESID>(a, it, lane, dts, max_out(a, a.imax_new));
}

// The books of a mirrored launch (HfStepArgs::mirrored), kept by its last
// workgroup; true for its waves.
template <class R>
__device__ __forceinline__ bool keeps_books(const HfStepArgs<R>& a)
{
    if (!a.mirrored || blockIdx.x != gridDim.x - 1) return false;
    for (int p = threadIdx.x; p < a.nprob; p += blockDim.x)
        a.calls_next[p] = a.calls[p] + (a.use_fixed ? 0u : (uint32_t)a.probs[p].cps);
    for (int i = threadIdx.x; i < a.nclear; i += blockDim.x) a.clear[i] = 0ull;
    if (threadIdx.x < HF_SYNC_WORDS) a.clear_sync[threadIdx.x] = 0u;
    if (threadIdx.x == 0 && a.fixstats) a.fixstats[0] += 1ull;   // launches of a context run one after the other
    return true;
}

template <class M, int LIM, bool RESID>
__global__ __launch_bounds__(256, 2) void k_muscl(const HfStepArgs<typename M::R> a)
{
    typedef typename M::R R;
    if (keeps_books(a)) return;
    const unsigned extra = a.mirrored ? 1u : 0u;
    const int lane = threadIdx.x & 63;
    int cached = -1;   // the block whose speculative dts this wave has computed
    double c_step = 0.0, c_pred = 0.0;
    long long c_kstep = 0, c_kpred = 0;
    // every item of the list, or with skipped blocks tickets over the
    // segments of the others
    const bool some = a.nskip && !a.use_fixed && __builtin_amdgcn_readfirstlane(*a.nskip) != 0u;
    const int nseg = 3 * a.nblocks;
    unsigned n = (unsigned)a.nmain;
    RangeCursor cur;
    if (some) {
        n = 0u;
        for (int c0 = 0; c0 < nseg; c0 += 64) {
            const int k = c0 + lane;
            const unsigned cnt = (k < nseg && !a.skip[k % a.nblocks]) ? (unsigned)a.segs[2 * k + 1] : 0u;
            unsigned tot;
            lane_prefix(cnt, tot);
            n += tot;
        }
        main_chunk<R>(a, cur, 0);
        cur.base = 0u;
    }
    for (unsigned t = ticket_first(n, extra); t < n; t = ticket_next(a.sync, lane, n, extra)) {
        unsigned idx = t;
        if (some) {
            while (t >= cur.base + cur.total) {
                const unsigned nb_ = cur.base + cur.total;
                if (cur.c0 + 64 >= nseg) return;   // not reached: the chunks hold n items
                main_chunk<R>(a, cur, cur.c0 + 64);
                cur.base = nb_;
            }
            int j;
            idx = cursor_item(cur, t, j);
            if (idx >= (unsigned)a.nmain) return;
        }
        main_item<M, LIM, RESID>(a, idx, lane, cached, c_step, c_pred, c_kstep, c_kpred);
    }
}

// The guess launch's view of problem p: its plan and the cursor over its
// blocks from the plan's first block on (a range per block: its items in the
// fix-up rounds, taken if the block needs computing).
struct GuessProblem {
    int p, first, nb;
    double O, m;
    long long kstep;
};

template <class R>
__device__ __forceinline__ bool guess_need(const HfStepArgs<R>& a, const GuessProblem& g, int c, int b)
{
    const double cf = cfl_eff(a.cfl, g.kstep + 1 + c);
    return a.skip[b] != 0u || cf * g.O != cf * smin(1e16, g.m);
}

template <class R>
__device__ __forceinline__ void guess_chunk(const HfStepArgs<R>& a, const GuessProblem& g, RangeCursor& cur, int c0)
{
    const int c = c0 + (int)(threadIdx.x & 63);
    cur.c0 = c0;
    cur.first = 0;
    cur.cnt = 0u;
    if (c >= g.first && c < g.nb) {
        const int b = a.probs[g.p].first + c;
        if (guess_need<R>(a, g, c, b)) {
            cur.first = a.fixrange[2 * b];
            cur.cnt = (unsigned)a.fixrange[2 * b + 1];
        }
    }
    cur.pre = lane_prefix(cur.cnt, cur.total);
}

// The next problem from p on with blocks to compute (nprob if none).
template <class R>
__device__ __forceinline__ void guess_enter(const HfStepArgs<R>& a, GuessProblem& g, int p)
{
    for (; p < a.nprob; p++) {
        const HfProbDev pr = a.probs[p];
        if (pr.nb < 2) continue;
        g.p = p;
        g.nb = pr.nb;
        g.first = guess_plan<R>(a, p, pr, g.O, g.m, g.kstep);
        if (g.first < pr.nb) return;
    }
    g.p = a.nprob;
}

template <class M, int LIM>
__global__ __launch_bounds__(256, 2) void k_muscl_guess(const HfStepArgs<typename M::R> a)
{
    typedef typename M::R R;
    const int lane = threadIdx.x & 63;
    // items to compute, over every problem; the walk below starts from the
    // first problem's first chunk, kept from this pass
    unsigned n = 0u;
    GuessProblem g, g0;
    RangeCursor cur;
    g0.p = a.nprob;
    for (guess_enter<R>(a, g, 0); g.p < a.nprob; guess_enter<R>(a, g, g.p + 1))
        for (int c0 = g.first & ~63; c0 < g.nb; c0 += 64) {
            RangeCursor ck;
            guess_chunk<R>(a, g, ck, c0);
            if (g0.p == a.nprob) {
                g0 = g;
                cur = ck;
            }
            n += ck.total;
        }
    if (n == 0u) return;
    g = g0;
    cur.base = 0u;
    int cb = -1;   // the block whose dts this wave holds
    double dt_step = 0.0, dt_pred = 0.0;
    long long kpred = 0;
    for (unsigned t = ticket_first(n); t < n; t = ticket_next(a.sync, lane, n)) {
        while (t >= cur.base + cur.total) {
            const unsigned nb_ = cur.base + cur.total;
            int c0 = cur.c0 + 64;
            if (c0 >= g.nb) {
                guess_enter<R>(a, g, g.p + 1);
                if (g.p >= a.nprob) return;   // not reached: the problems hold n items
                c0 = g.first & ~63;
            }
            guess_chunk<R>(a, g, cur, c0);
            cur.base = nb_;
        }
        int j;
        const unsigned idx = cursor_item(cur, t, j);
        if (idx < (unsigned)a.nmain || idx >= (unsigned)a.nitems) return;
        const HfItem it = a.items[a.item0 + idx];
        const HfBlockDev bd = a.blocks[it.block];
        if (it.block != cb) {
            cb = it.block;
            kpred = g.kstep + 1 + bd.lb;
            dt_step = cfl_eff(a.cfl, g.kstep) * g.O;
            dt_pred = cfl_eff(a.cfl, kpred) * smin(1e16, g.m);
            a.fixed[cb] = 1u;   // the same value from every wave
        }
        record_dts<R>(a, it, bd, false, dt_step, dt_pred, g.kstep, kpred);
        auto dts = [&](double& step, double& pred) { step = dt_step; pred = dt_pred; };
        muscl_go<M, LIM, false>(a, it, lane, dts, max_out(a, a.imax_fix));
    }
}

template <class M, int LIM>
__global__ __launch_bounds__(256, 2) void k_muscl_check(const HfStepArgs<typename M::R> a)
{
    typedef typename M::R R;
    const int lane = threadIdx.x & 63;
    // the first round with a wrong block; wave 0 records the skip verdicts
    int first = a.nrounds + 1;
    const bool rec = wave_id() == 0;
    Verdict v;
    for (int p = 0; p < a.nprob; p++) {
        const HfProbDev pr = a.probs[p];
        if (pr.nb < 2) continue;
        double O;
        PlanTerms t;
        v.problem = p;
        guess_plan<R>(a, p, pr, O, v.mg, v.kstep, t);
        const int w = plan_scan<R, PRE_GUESS>(a, pr, a.nblocks, v.kstep, O, t, v.mg, rec);
        first = w < first ? w : first;
    }
    if (first > a.nrounds) return;   // every block has its exact dt

    // one round computes at a time: more waves than the largest has items would
    // only draw tickets and poll (8 x 97^2 channel, 194 items a round: 160 us a
    // launch with all 2 048, now 80)
    unsigned waves = 0u;
    for (int l = first; l <= a.nrounds; l++) waves = max(waves, (unsigned)(a.rounds[l + 1] - a.rounds[l]));
    waves = min(waves, total_waves());
    if (wave_id() >= waves) return;

    const MaxOut imax_chk = {a.imax_fix + HF_MAX_SLOT(a.nblocks, 0, a.ways, a.way_stride), 0};
    uint32_t* fixed_chk = a.fixed + a.nblocks;
    const unsigned base = (unsigned)a.rounds[first];   // item of queue counter value 0
    int r_from = -1, r_busy = 0;   // first_busy_round(r_from) as this wave last computed it
    for (unsigned idx = next_ticket(a.sync, lane, base);; idx = next_ticket(a.sync, lane, base)) {
        if (idx >= (unsigned)a.nitems) break;
        const HfItem it = a.items[a.item0 + idx];
        const int l = round_of<R>(a, idx);
        if (l != r_from) {
            if (!wait_done(a.sync, (unsigned)a.rounds[l] - base, a.wait_ticks)) {
                const unsigned k = idx - (unsigned)a.nmain;
                atomicOr(&a.pending[k >> 5], 1u << (k & 31));
                continue;   // left to the last wave, not counted complete
            }
            r_from = l;
            r_busy = first_busy_round<R>(a, l, lane, base, v);
        }
        if (r_busy == l) {
            const HfBlockDev bd = a.blocks[it.block];
            if (it.block != v.block) {
                const HfProbDev pr = a.probs[bd.problem];
                verdict_on<R>(a, bd.problem, pr, bd.lb, v);
            }
            if (v.need) {
                // Or, not an exchange: the compiler leaves one lane's of an or
                // with one value for the wave, and 64 of an exchange, which
                // took 1.3 ms of the 1.5 ms a recomputed 1024^2 block cost
                // (the channel's first 200 steps: 2.9 -> 0.83 ms per step).
                atomicOr(&fixed_chk[it.block], 1u);
                record_dts<R>(a, it, bd, false, v.step, v.pred, v.kstep, v.kpred);
                auto dts = [&](double& step, double& pred) { step = v.step; pred = v.pred; };
                muscl_go<M, LIM, false>(a, it, lane, dts, imax_chk);
            }
        }
        item_done(a.sync, lane);
    }
    // The last wave to leave computes the items whose wait gave up, in queue
    // order; every other wave has left, so all it reads is final, and none of
    // those items was written by another wave.
    __builtin_amdgcn_s_waitcnt(0xF70);   // this wave's atomics are performed before it counts as gone
    const unsigned left = __builtin_amdgcn_readfirstlane(atomicAdd(&a.sync[HF_SYNC_EXITED], lane == 0 ? 1u : 0u));
    if (left != waves - 1) return;
    if (!(__builtin_amdgcn_readfirstlane(coherent_read(&a.sync[HF_SYNC_DONE])) & HF_SYNC_ABORT_BIT)) return;
    const unsigned nfix = (unsigned)(a.nitems - a.nmain);
    for (unsigned w = 0; w * 32 < nfix; w++) {
        const unsigned bits = __builtin_amdgcn_readfirstlane(coherent_read(&a.pending[w]));
        for (unsigned k = 0; k < 32; k++) {
            if (!((bits >> k) & 1u)) continue;
            const unsigned idx = a.nmain + w * 32 + k;
            const HfItem it = a.items[a.item0 + idx];
            const HfBlockDev bd = a.blocks[it.block];
            const HfProbDev pr = a.probs[bd.problem];
            verdict_on<R>(a, bd.problem, pr, bd.lb, v);
            if (v.need) {
                atomicOr(&fixed_chk[it.block], 1u);
                record_dts<R>(a, it, bd, false, v.step, v.pred, v.kstep, v.kpred);
                auto dts = [&](double& step, double& pred) { step = v.step; pred = v.pred; };
                muscl_go<M, LIM, false, false>(a, it, lane, dts, imax_chk);   // rare: the general rows only
                __builtin_amdgcn_s_waitcnt(0xF70);   // its maxima are performed before the next verdict reads them
            }
        }
        atomicExch(&a.pending[w], 0u);
    }
}

// ---------------------------------------------------------------- Godunov --
// Rows of a Godunov item in range, as muscl_rows_q64.
template <class M, class DtOf>
__device__ __forceinline__ int godunov_rows_q64(const HfStepArgs<double>& a, const HfItem it, const HfBlockDev& bd,
                                                const int lane, DtOf&& dt_of, double& dt, double& mx, double& my)
{
    const double gam = a.gamma, g1 = a.gamma - 1.0;
    const int xraw = it.x0 + lane;
    const bool valid = xraw < bd.tx;
    const int xc = valid ? xraw : bd.tx - 1;
    const Lines<double, false> ROW(a, bd, xc);
    const int pitch = bd.pitch, ty = bd.ty;
    const int64_t plane = bd.plane;
    const bool out = valid && lane >= 1 && lane < 63 && xraw >= 1 && xraw < bd.tx - 1;
    const q64::mask m0 = __ballot(out), m1 = m0 | m0 << 1 | m0 >> 1;   // lanes that write, and their x neighbours
    const int y0 = it.y0;
    double ub[4], uc[4], un[4], Gs[4];
    const unsigned fb = ROW(y0 - 1, ub), fc = ROW(y0, uc);
    unsigned fn = ROW(y0 + 1, un);
    ROW.signed_line(ub, fb);
    ROW.signed_line(uc, fc);
    const double ig1 = 1.0 / g1, rdx = 1.0 / bd.dx, rdy = 1.0 / bd.dy;
    const q64::Limits lim;
    q64::mask bad = q64::out_of_range(ub, lim), bc = q64::out_of_range(uc, lim);
    q64::State sc;
    if ((bad | bc) & m0) {   // before arithmetic that would be done twice
        bad = m0;
    } else {
        sc = q64::make_state(uc, gam, g1, ig1, bc, lim);
        const q64::State sb = q64::make_state(ub, gam, g1, ig1, bad, lim);
        q64::hllc<false>(sb, sc, Gs, bad, lim);         // face y0-1/2
    }
    dt = dt_of();
    if (!q64::constants_in_range(gam, g1) || (bad & m0)) return 0;
    double* Ob = a.O + bd.off;
    for (int r = 0; r < it.rows; r++) {
        const int y = y0 + r;
        double nn[4];
        ROW.signed_line(un, fn);
        fn = ROW(y + 2 < ty ? y + 2 : ty - 1, nn);     // next iteration's U(y+1)
        q64::mask bn = q64::out_of_range(un, lim), bx = 0;
        const q64::State sn = q64::make_state(un, gam, g1, ig1, bn, lim);
        double Gn[4], Fw[4], Fe[4];
        q64::hllc<false>(sc, sn, Gn, bn, lim);          // face y+1/2

        q64::State sw;
        sw.U0 = shfl_up1(sc.U0); sw.U1 = shfl_up1(sc.U1); sw.U2 = shfl_up1(sc.U2); sw.U3 = shfl_up1(sc.U3);
        sw.u = shfl_up1(sc.u); sw.v = shfl_up1(sc.v); sw.p = shfl_up1(sc.p); sw.E = shfl_up1(sc.E);
        sw.a = shfl_up1(sc.a); sw.y = shfl_up1(sc.y);
        q64::hllc<true>(sw, sc, Fw, bx, lim);           // face x-1/2
        for (int k = 0; k < 4; k++) Fe[k] = shfl_dn1(Fw[k]);

        const double U[4] = {sc.U0, sc.U1, sc.U2, sc.U3};
        double Ln[4], Un[4], dx_, dy_;
        update_cell<M>(rdx, rdy, dt, Fw, Fe, Gs, Gn, U, Ln, Un);
        q64::mask bw = 0;
        q64::wave_speeds(Un, gam, g1, dx_, dy_, bw, lim);
        if (((bn | bw) & m0) | ((bc | bx) & m1)) return r;
        if (out) {
            double* o = Ob + (int64_t)y * pitch + xraw;
            for (int k = 0; k < 4; k++) o[k * plane] = Un[k];
            mx = dmax_nan(mx, dx_);
            my = dmax_nan(my, dy_);
        }
        for (int k = 0; k < 4; k++) { Gs[k] = Gn[k]; un[k] = nn[k]; }
        sc = sn;
        bc = bn;
    }
    return it.rows;
}

// GodunovScheme::operator() (scheme/godunov/godunov.cpp:27-118) fused with
// the forward Euler update.  Each cell's primitives and sound speed are
// computed once and shared by its four faces.  Output columns per wave: 62.
// dt_of() gives the step's dt; it is called after the item's first rows are
// requested and the first face flux computed, none of which needs the dt,
// so the dt's chain of dependent loads overlaps their memory latency.
template <class M, bool RESID, class DtOf>
__device__ __forceinline__ void godunov_item(const HfStepArgs<typename M::R>& a, const HfItem it, const int lane,
                                             DtOf&& dt_of, const MaxOut& imax_out)
{
    typedef typename M::R R;

    const HfBlockDev bd = a.blocks[it.block];
    const int xraw = it.x0 + lane;
    const bool valid = xraw < bd.tx;
    const int xc = valid ? xraw : bd.tx - 1;
    const Lines<R, false> ROW(a, bd, xc);
    const int pitch = bd.pitch, ty = bd.ty;
    const int64_t plane = bd.plane;
    const bool out = valid && lane >= 1 && lane < 63 && xraw >= 1 && xraw < bd.tx - 1;

    const R rdx = R(1.0 / bd.dx);                  // godunov.cpp:97-98
    const R rdy = R(1.0 / bd.dy);
    const R gam = R(a.gamma), g1 = R(a.gamma - 1.0);

    double mx = 0.0, my = 0.0, dt = 0.0;
    int done = 0;
    constexpr bool QUICK = !RESID && !M::fast;
    if constexpr (QUICK) done = godunov_rows_q64<M>(a, it, bd, lane, dt_of, dt, mx, my);
    if (done < it.rows) {
    const int y0 = it.y0 + done, rows = it.rows - done;
    R ub[4], uc[4], un[4];
    const unsigned fb = ROW(y0 - 1, ub), fc = ROW(y0, uc);
    unsigned fn = ROW(y0 + 1, un);                 // loaded one iteration ahead
    ROW.signed_line(ub, fb);
    ROW.signed_line(uc, fc);
    State<R> sb = make_state<M>(ub, gam, g1);
    State<R> sc = make_state<M>(uc, gam, g1);
    R Gs[4];
    hllc<M, false>(sb, sc, Gs);                    // face y0-1/2
    const R dtR = QUICK ? R(dt) : R(dt_of());
    R* Ob = RESID ? a.O : a.O + bd.off;
    for (int r = 0; r < rows; r++) {
        const int y = y0 + r;
        R nn[4];
        ROW.signed_line(un, fn);
        fn = ROW(y + 2 < ty ? y + 2 : ty - 1, nn);     // next iteration's U(y+1)
        const State<R> sn = make_state<M>(un, gam, g1);
        R Gn[4], Fw[4], Fe[4];
        hllc<M, false>(sc, sn, Gn);                // face y+1/2

        State<R> sw;
        sw.U0 = shfl_up1(sc.U0); sw.U1 = shfl_up1(sc.U1); sw.U2 = shfl_up1(sc.U2); sw.U3 = shfl_up1(sc.U3);
        sw.u = shfl_up1(sc.u); sw.v = shfl_up1(sc.v); sw.p = shfl_up1(sc.p); sw.E = shfl_up1(sc.E);
        sw.a = shfl_up1(sc.a);
        hllc<M, true>(sw, sc, Fw);                 // face x-1/2
        for (int k = 0; k < 4; k++) Fe[k] = shfl_dn1(Fw[k]);

        const R U[4] = {sc.U0, sc.U1, sc.U2, sc.U3};
        R Ln[4], Un[4];
        update_cell<M>(rdx, rdy, dtR, Fw, Fe, Gs, Gn, U, Ln, Un);
        if (out) {
            R* o = Ob + (int64_t)y * pitch + xraw;
            for (int k = 0; k < 4; k++) o[k * plane] = RESID ? Ln[k] : Un[k];
            if (!RESID) {
                double dx_, dy_;
                wave_speeds<M>(Un[0], Un[1], Un[2], Un[3], gam, g1, dx_, dy_);
                mx = dmax_nan(mx, dx_);
                my = dmax_nan(my, dy_);
            }
        }
        for (int k = 0; k < 4; k++) { Gs[k] = Gn[k]; un[k] = nn[k]; }
        sc = sn;
    }
    }
    if (!RESID) store_maxima(a, imax_out, it.block, wave_max(mx), wave_max(my));
}

// Persistent Godunov launch (no predictor, so never a fix-up).
template <class M, bool RESID>
__global__ __launch_bounds__(256) void k_godunov(const HfStepArgs<typename M::R> a)
{
    typedef typename M::R R;
    if (keeps_books(a)) return;
    const unsigned extra = a.mirrored ? 1u : 0u;
    const int lane = threadIdx.x & 63;
    const unsigned n = (unsigned)a.nitems;
    for (unsigned idx = ticket_first(n, extra); idx < n; idx = ticket_next(a.sync, lane, n, extra)) {
        const HfItem it = a.items[a.item0 + idx];
        auto dt_of = [&]() -> double {
            if (a.use_fixed) return a.fixed_step;
            const HfBlockDev bd = a.blocks[it.block];
            double dt_step, dt_pred;
            long long kstep, kpred;
            step_dts<R>(a, bd, false, dt_step, dt_pred, kstep, kpred);
            const long long hs = kstep - a.hist_base;
            if (bd.problem == 0 && bd.lb == 0 && it.x0 == 0 && it.y0 == bd.g && hs >= 1 && hs <= a.hist_cap)
                a.hist[hs - 1] = dt_step;
            return dt_step;
        };
        godunov_item<M, RESID>(a, it, lane, dt_of, max_out(a, a.imax_new));
    }
}

// ------------------------------------------------------------- ghost fill --
// Mesh::apply_bcs (mesh/mesh/mesh.cpp:31-39) as a gather: the host replays the
// reference's sequential side order symbolically and records, for every
// ghost cell, which pre-fill cell (or Dirichlet constant) it ends up holding
// and which momentum components were negated on the way.  Reads come from S,
// writes go to D, so the fill is race-free in one launch.  Also reduces the
// ghosts' max wave speeds per block, and (step mode, in one extra workgroup
// after those of the ghost cells) advances each problem's TimeStep call
// counter and clears the partial maxima of the next step.

constexpr int GHOST_WAVES = 4;   // k_ghost workgroups: 256 threads
template <class M>
__global__ __launch_bounds__(256) void k_ghost(const HfGhost* __restrict__ tab, int n,
                                               const HfBlockDev* __restrict__ blocks,
                                               const typename M::R* __restrict__ S, typename M::R* __restrict__ D,
                                               const typename M::R* __restrict__ consts, unsigned long long* gmax,
                                               double gamma, GhostBook book)
{
    typedef typename M::R R;
    // The last workgroup keeps the step's books (none of it reads or writes a
    // ghost cell or gmax), beside the ghost cells instead of ahead of some.
    if (blockIdx.x == gridDim.x - 1) {
        for (int p = threadIdx.x; p < book.nprob && book.bump; p += blockDim.x)
            book.calls[p] += (uint32_t)book.probs[p].cps;
        for (int i = threadIdx.x; i < book.nclear0; i += blockDim.x) book.clear0[i] = 0ull;
        for (int i = threadIdx.x; i < book.nclear1; i += blockDim.x) book.clear1[i] = 0ull;
        for (int i = threadIdx.x; i < book.nturn; i += blockDim.x) {
            unsigned long long* const t = book.turns + i;
            t[0] = t[(int64_t)book.turn * book.nturn];
            t[book.nturn] = 0ull;
            t[2 * (int64_t)book.nturn] = 0ull;
        }
        for (int i = threadIdx.x; i < book.nqueue; i += blockDim.x) book.queue[i] = 0u;
        for (int i = threadIdx.x; i < book.npending; i += blockDim.x) book.pending[i] = 0u;
        const int nb = book.nblocks, bw = book.block_words;
        // the check launch's recomputation over the guess launch's
        for (int i = threadIdx.x; i < nb * bw && book.fixed; i += blockDim.x) {
            const int b = i / bw;
            const int s = book.fixed[nb + b] ? 1 : book.fixed[b] ? 0 : -1;
            if (s >= 0) book.imax_prev[i] = book.imax_fix[s * nb * bw + i];
            book.imax_fix[i] = 0ull;
            book.imax_fix[nb * bw + i] = 0ull;
        }
        __syncthreads();   // the fixed flags are read; the skip count below starts from zero
        if (book.fixstats && book.fixed && threadIdx.x == 0) atomicAdd(&book.fixstats[0], 1ull);
        for (int b = threadIdx.x; b < nb && book.fixed; b += blockDim.x) {
            if (book.fixstats) {
                if (book.skip[b]) atomicAdd(&book.fixstats[1], 1ull);
                if (book.fixed[b]) atomicAdd(&book.fixstats[2], 1ull);
                if (book.fixed[nb + b]) atomicAdd(&book.fixstats[3], 1ull);
            }
            book.skip[b] = book.skip_next[b];
            if (book.skip_next[b]) atomicAdd(&book.queue[HF_SLOT_MAIN * HF_SYNC_WORDS + HF_SYNC_NSKIP], 1u);
            for (int t = 0; t < 2; t++) book.fixed[t * nb + b] = 0u;
        }
        return;
    }
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    double dx_ = 0.0, dy_ = 0.0;
    int blk = -1;
    if (gid < n) {
        const HfGhost e = tab[gid];
        R u[4];
        if (e.src_block >= 0) {
            const HfBlockDev sb = blocks[e.src_block];
            const R* p = S + sb.off + (e.src_cell & HF_CELL_MASK);
            load_cell<R>(p, sb.plane, u);
        } else {
            const R* c = consts + 4 * (-e.src_block - 1);
            u[0] = c[0]; u[1] = c[1]; u[2] = c[2]; u[3] = c[3];
        }
        if (e.src_cell & HF_FLIP_U) u[1] = -u[1];
        if (e.src_cell & HF_FLIP_V) u[2] = -u[2];
        const HfBlockDev db = blocks[e.dst_block];
        R* q = D + db.off + e.dst_cell;
        q[0] = u[0];
        q[db.plane] = u[1];
        q[2 * db.plane] = u[2];
        q[3 * db.plane] = u[3];
        double x, y;
        wave_speeds<M>(u[0], u[1], u[2], u[3], R(gamma), R(gamma - 1.0), x, y);
        dx_ = dmax_nan(0.0, x);
        dy_ = dmax_nan(0.0, y);
        blk = e.dst_block;
    }
    // The table is grouped by destination block: a wave covering one block
    // reduces to one value, and thread 0 merges consecutive waves of the same
    // block, so a workgroup issues one atomic per block it covers (device-
    // scope atomics on one address serialise: one per wave made this launch
    // take 20 us on 66 k ghost cells, one per workgroup 13 us; reading the
    // slot first made it slower still).  A wave spanning two blocks uses
    // per-lane atomics.
    __shared__ int wblk[GHOST_WAVES];
    __shared__ double wmx[GHOST_WAVES], wmy[GHOST_WAVES];
    const int w = threadIdx.x >> 6;
    const int b0 = __shfl(blk, 0, 64);
    const bool uniform = __all(blk == b0 || blk < 0);
    if (uniform) {
        const double wx = wave_max(dx_), wy = wave_max(dy_);
        if (lane == 0) {
            wblk[w] = b0;
            wmx[w] = wx;
            wmy[w] = wy;
        }
    } else {
        if (blk >= 0) {
            atomicMax(&gmax[2 * blk], dbits(dx_));
            atomicMax(&gmax[2 * blk + 1], dbits(dy_));
        }
        if (lane == 0) wblk[w] = -1;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int cb = -1;
        double cx = 0.0, cy = 0.0;
        for (int k = 0; k < (int)(blockDim.x >> 6); k++) {
            if (wblk[k] == cb) {
                cx = (wmx[k] > cx) ? wmx[k] : cx;
                cy = (wmy[k] > cy) ? wmy[k] : cy;
                continue;
            }
            if (cb >= 0) {
                atomicMax(&gmax[2 * cb], dbits(cx));
                atomicMax(&gmax[2 * cb + 1], dbits(cy));
            }
            cb = wblk[k];
            cx = wmx[k];
            cy = wmy[k];
        }
        if (cb >= 0) {
            atomicMax(&gmax[2 * cb], dbits(cx));
            atomicMax(&gmax[2 * cb + 1], dbits(cy));
        }
    }
}

// -------------------------------------------------------------- wave scan --
// Max of |u|+c and |v|+c over cells of blocks (TimeStep::operator(),
// timestep.cpp:37-55), one workgroup per item (rows [y0, y0 + rows) of a
// block, lanes along x, a wave per row): interior cells are read from I, ghost
// cells from Gh; with interior_only the ghosts are skipped.  Reads each value
// once; HBM bounds it.  One atomic pair per workgroup, on the block's slots:
// with one per wave on one word the scan of 1024^2 FP64 cells took 375 us, of
// 8192^2 FP32 506, of 512 blocks (a launch each) 17 ms; now 20, 331 and 166 us.
template <class M>
__global__ __launch_bounds__(256) void k_scan(const HfItem* __restrict__ items, const HfBlockDev* __restrict__ blocks,
                                              const typename M::R* __restrict__ I,
                                              const typename M::R* __restrict__ Gh, int interior_only, double gamma,
                                              unsigned long long* outmax, int ways, int stride)
{
    typedef typename M::R R;
    const HfItem it = items[blockIdx.x];
    const HfBlockDev bd = blocks[it.block];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double mx = 0.0, my = 0.0;
    for (int y = it.y0 + w; y < it.y0 + it.rows; y += 4) {
        const bool gy = y < bd.g || y >= bd.ty - bd.g;
        if (gy && interior_only) continue;
        const int64_t row = bd.off + (int64_t)y * bd.pitch;
#pragma unroll 4
        for (int x = lane; x < bd.tx; x += 64) {
            const bool gh = gy || x < bd.g || x >= bd.tx - bd.g;
            if (gh && interior_only) continue;
            R u[4];
            load_cell<R>((gh ? Gh : I) + row + x, bd.plane, u);
            double dx_, dy_;
            wave_speeds<M>(u[0], u[1], u[2], u[3], R(gamma), R(gamma - 1.0), dx_, dy_);
            mx = dmax_nan(mx, dx_);
            my = dmax_nan(my, dy_);
        }
    }
    __shared__ double sx[4], sy[4];
    mx = wave_max(mx);
    my = wave_max(my);
    if (lane == 0) {
        sx[w] = mx;
        sy[w] = my;
    }
    __syncthreads();
    if (threadIdx.x < 2) {   // thread 0: x, thread 1: y
        const double* s = threadIdx.x == 0 ? sx : sy;
        double m = s[0];
        for (int k = 1; k < 4; k++) m = s[k] > m ? s[k] : m;
        atomicMax(outmax + HF_MAX_SLOT(it.block, blockIdx.x & (ways - 1), ways, stride) + threadIdx.x, dbits(m));
    }
}

// n values of a block's dense [4][ty][tx] form from value x0 of row row0 on,
// in binary64: src is the block's padded planes, dst pinned host memory (the
// link bounds it).
template <class R>
__global__ __launch_bounds__(256) void k_dense(const R* __restrict__ src, int64_t plane, int pitch, uint32_t tx,
                                               uint32_t ty, uint32_t row0, uint32_t x0, uint32_t n, double* dst)
{
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const uint32_t t = x0 + i, row = row0 + t / tx, x = t % tx;
        dst[i] = (double)src[(row / ty) * plane + (int64_t)(row % ty) * pitch + x];
    }
}

// --------------------------------------------------- conservation sums --
// Neumaier-compensated FP64 partial sums of the four conserved variables
// over a block's interior; one (sum, compensation) pair per workgroup and
// variable, combined on the host in workgroup order.
template <class R>
__global__ __launch_bounds__(256) void k_conserve(HfBlockDev bd, const R* __restrict__ A, double* part)
{
    __shared__ double ss[4][256];
    __shared__ double cc[4][256];
    double s[4] = {0, 0, 0, 0}, c[4] = {0, 0, 0, 0};
    const int64_t n = (int64_t)bd.nx * bd.ny;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int y = (int)(i / bd.nx) + bd.g, x = (int)(i % bd.nx) + bd.g;
        const R* p = A + bd.off + (int64_t)y * bd.pitch + x;
        for (int k = 0; k < 4; k++) {
            const double v = (double)p[k * bd.plane];
            const double t = s[k] + v;
            c[k] += (__builtin_fabs(s[k]) >= __builtin_fabs(v)) ? ((s[k] - t) + v) : ((v - t) + s[k]);
            s[k] = t;
        }
    }
    for (int k = 0; k < 4; k++) { ss[k][threadIdx.x] = s[k]; cc[k][threadIdx.x] = c[k]; }
    __syncthreads();
    if (threadIdx.x < 4) {
        const int k = threadIdx.x;
        double S = 0.0, Cm = 0.0;
        for (int i = 0; i < (int)blockDim.x; i++) {
            const double v = ss[k][i];
            const double t = S + v;
            Cm += (__builtin_fabs(S) >= __builtin_fabs(v)) ? ((S - t) + v) : ((v - t) + S);
            S = t;
            Cm += cc[k][i];
        }
        part[(blockIdx.x * 4 + k) * 2] = S;
        part[(blockIdx.x * 4 + k) * 2 + 1] = Cm;
    }
}

}  // namespace hf
