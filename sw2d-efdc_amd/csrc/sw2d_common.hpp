// sw2d_common.hpp -- device code shared by the fused and the plain kernels:
// iteration timing, forcing evaluation, wave reductions, the bookkeeping
// (clock ring, volume ledger, hydrograph, lake-inflow integration).
#pragma once
#include "sw2d_internal.hpp"
#include "sw2d_math.hpp"

namespace sw2d {

struct StepTime {
    double t, dt, dt2, tm;
};

// Wave-wide reductions with a fixed combination order: lane i with lane i ^ 32,
// then ^ 16 and so on (lane 0 holds the result; all lanes active).  The halves of
// the wave and of its half rows are brought together by lane swaps, the rest by
// DPP moves within rows of 16: after ^ 8 a row repeats itself, so a rotation by
// 4 is ^ 4.  LDS permutes in their place wait for LDS six times a value.
__device__ __forceinline__ int lane_hi(double v) { return (int)((unsigned long long)__double_as_longlong(v) >> 32); }
__device__ __forceinline__ int lane_lo(double v) { return (int)__double_as_longlong(v); }
__device__ __forceinline__ double lane_double(unsigned hi, unsigned lo)
{
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
template <int CTRL> __device__ __forceinline__ double dpp_row(double v)
{
    return lane_double(__builtin_amdgcn_update_dpp(0, lane_hi(v), CTRL, 0xf, 0xf, true),
                       __builtin_amdgcn_update_dpp(0, lane_lo(v), CTRL, 0xf, 0xf, true));
}
// f(own, other) over a row of 16 lanes whose values it combines
template <typename Op> __device__ __forceinline__ double row_reduce(double v, const Op &f)
{
    v = f(v, dpp_row<0x128>(v));  // row_ror:8
    v = f(v, dpp_row<0x124>(v));  // row_ror:4
    v = f(v, dpp_row<0x4e>(v));   // quad_perm [2, 3, 0, 1]
    return f(v, dpp_row<0xb1>(v));  // quad_perm [1, 0, 3, 2]
}
template <typename Op> __device__ __forceinline__ double wave_reduce(double v, const Op &f)
{
    {
        const auto h = __builtin_amdgcn_permlane32_swap(lane_hi(v), lane_hi(v), false, false);
        const auto l = __builtin_amdgcn_permlane32_swap(lane_lo(v), lane_lo(v), false, false);
        v = f(lane_double(h[0], l[0]), lane_double(h[1], l[1]));
    }
    {
        const auto h = __builtin_amdgcn_permlane16_swap(lane_hi(v), lane_hi(v), false, false);
        const auto l = __builtin_amdgcn_permlane16_swap(lane_lo(v), lane_lo(v), false, false);
        v = f(lane_double(h[0], l[0]), lane_double(h[1], l[1]));
    }
    return row_reduce(v, f);
}
__device__ __forceinline__ double wave_sum(double v)
{
    return wave_reduce(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double wave_max(double v)
{
    return wave_reduce(v, [](double a, double b) { return (b > a) ? b : a; });
}
__device__ __forceinline__ double wave_min(double v)
{
    return wave_reduce(v, [](double a, double b) { return (b < a) ? b : a; });
}

// the CFL minimum of a clock slot: one partial minimum a lane, combined over
// the wave (all lanes active; the result is the same in every lane)
__device__ __forceinline__ double clock_cfl(const Clock &ck)
{
    static_assert(kCflSlots == 16, "a row of lanes");
    const double m = row_reduce(__longlong_as_double((long long)ck.cfl[threadIdx.x & (kCflSlots - 1)].bits),
                                [](double a, double b) { return (b < a) ? b : a; });
    const long long b = __double_as_longlong(m);  // uniform: into scalar registers
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
// folds one wave's CFL minimum into it; i: any number that spreads the waves
__device__ __forceinline__ void clock_note_cfl(Clock &ck, int i, double cfl)
{
    atomicMin(&ck.cfl[i & (kCflSlots - 1)].bits, (unsigned long long)__double_as_longlong(cfl));
}

// start time and length of this iteration from the clock ring; ADAPT false:
// the step is known to be fixed
template <bool ADAPT = true>
__device__ __forceinline__ StepTime step_time(const StepCommon &s, const Iter &it)
{
    const Clock &ck = s.clk[it.slot_a];
    StepTime st;
    st.t = ck.t;
    if (!ADAPT || s.fixed_dt) {
        st.dt = s.dt_fixed;
        st.dt2 = s.dt2_fixed;
    } else {
        double d = s.courant * clock_cfl(ck);
        st.dt2 = (d < s.dt2_max) ? d : s.dt2_max;
        st.dt = 0.5 * st.dt2;
    }
    st.tm = st.t + st.dt;
    return st;
}

// rr of stream_flow in m/s (SW2D-EFDC.cu:546-553); 0 without a rain series
__device__ __forceinline__ double rain_rate(const StepCommon &s, double t)
{
    if (s.nrain <= 0) return 0.0;
    double rr = series_value(s.rain, s.nrain, s.dtrain, t);
    return rr / (s.dtrain * 1000.0);
}

// Ev of evaporation_load in m/s (SW2D-EFDC.cu:588-600)
__device__ __forceinline__ double evap_rate(const StepCommon &s, double t)
{
    if (!s.evap_on) return 0.0;
    double e = series_value(s.evapo, s.nevapo, s.dtrain, t);
    return e / (s.dtrain * 1000.0);
}

// ql of source i in m/s (SW2D-EFDC.cu:531-539)
__device__ __forceinline__ double source_rate(const StepCommon &s, int i, double t)
{
    double ql = source_value(s.Q, s.nq, s.nst, i, s.dtoq, t);
    return ql / (s.dx * s.dy);
}

// uniform number in [0, 1) from (cell, iteration): a 32-bit integer hash
// (multiply-xorshift finaliser), 24 bits of it scaled by 2^-24
__device__ __forceinline__ float cell_uniform(uint32_t cell, uint32_t iter)
{
    uint32_t x = cell * 0x9E3779B1u ^ iter * 0x85EBCA77u;
    x ^= x >> 16;
    x *= 0x7FEB352Du;
    x ^= x >> 15;
    x *= 0x846CA68Bu;
    x ^= x >> 16;
    return (float)(x >> 8) * 5.9604644775390625e-08f;
}

// one factor of the moving Gaussian storm
__device__ __forceinline__ double storm_factor(double d, double sigma)
{
    return exp_d(-(d * d) / (2.0 * sigma * sigma));
}

__device__ __forceinline__ bool storm_live(const StepCommon &s, double t)
{
    return s.storm_on && (t >= s.st_t0) && (t < s.st_t1);
}

// inflow rate of one coupling record (couple_BC_efdc, SW2D-EFDC.cu:764-821)
__device__ __forceinline__ double bc_rate(int kind, double h, double uua, double vva, double dx,
                                          double dy)
{
    switch (kind) {
    case 0: return (uua < 0) ? -uua * h * dx : 0.00;
    case 1: return (uua > 0) ? uua * h * dx : 0.00;
    case 2: return (vva < 0) ? -vva * h * dy : 0.00;
    default: return (vva > 0) ? vva * h * dy : 0.00;
    }
}

// Face velocities of a state held in a pitched (rows x pitch) layout, with the
// reference's edge rules (hm_hn 362-398, uu1_vv1 404-452): every face outside
// the grid, on row 0 and on column 0 carries zero flux.  T is the type of the
// fluxes, TH that of the depths (the mixed form keeps depths in FP64): the
// face depth and its dry test are taken in TH, the velocity in T.
template <typename T, typename TH = T>
struct PitchedState {
    const TH *h;
    const T *um, *vn;
    int R, C, P;
    TH th;
    __device__ __forceinline__ TH hv(int r, int j) const { return h[(long)r * P + j]; }
    __device__ __forceinline__ T uu1(int r, int j) const
    {
        if (r <= 0 || r >= R || j < 0 || j >= C) return T(0);
        TH hm = TH(0.50) * (hv(r, j) + hv(r - 1, j));
        return (hm >= th) ? um[(long)r * P + j] / (T)hm : T(0.00);
    }
    __device__ __forceinline__ T vv1(int r, int j) const
    {
        if (r < 0 || r >= R || j <= 0 || j >= C) return T(0);
        TH hn = TH(0.50) * (hv(r, j) + hv(r, j - 1));
        return (hn >= th) ? vn[(long)r * P + j] / (T)hn : T(0.0);
    }
    // uua_vva, SW2D-EFDC.cu:489-522
    __device__ __forceinline__ T uua(int r, int j) const
    {
        if (j > 0) return T(0.250) * (uu1(r, j) + uu1(r + 1, j) + uu1(r, j - 1) + uu1(r + 1, j - 1));
        return T(0.50) * (uu1(r, j) + uu1(r + 1, j));
    }
    __device__ __forceinline__ T vva(int r, int j) const
    {
        if (r > 0) return T(0.250) * (vv1(r, j) + vv1(r, j + 1) + vv1(r - 1, j) + vv1(r - 1, j + 1));
        return T(0.50) * (vv1(r, j) + vv1(r, j + 1));
    }
};

// Bookkeeping of iteration k, one wave a part.  Part 0: advance the clock ring
// and (forcing) evaluate the next iteration's forcing.  Part 1: reduce the
// partial sums of iteration k-1 into the ledger (fixed order) and record its
// hydrograph sample.  Part b >= 2: integrate the lake inflow of records
// 64(b-2) .. 64b-65 over the state at the start of iteration k.  uua/vva are
// evaluated by the functor F.
__device__ __forceinline__ void reduce_partials(const Partial *p, int n, int lane, double &vol,
                                                double &src, double &clip, double &qo)
{
    vol = 0; src = 0; clip = 0; qo = 0;
    // One wave, so the latency of its loads is all there is: kInFlight records
    // a lane are asked for before the first is added (past the end: record
    // 0, added as zeros), in the order of one record after the other.
    constexpr int kInFlight = 8;
    for (int i = lane; i - lane < n; i += 64 * kInFlight) {
        Partial a[kInFlight];
#pragma unroll
        for (int c = 0; c < kInFlight; c++) a[c] = p[i + 64 * c < n ? i + 64 * c : 0];
#pragma unroll
        for (int c = 0; c < kInFlight; c++) {
            const bool in = i + 64 * c < n;
            vol += in ? a[c].vol : 0.0;
            src += in ? a[c].src : 0.0;
            clip += in ? a[c].clip : 0.0;
            qo += in ? a[c].qout : 0.0;
        }
    }
    vol = wave_sum(vol); src = wave_sum(src); clip = wave_sum(clip); qo = wave_sum(qo);
}

// Forcing of an iteration that starts at t, one value a lane: every wave of the
// iteration needs the same few numbers, each the end of a chain of dependent
// loads and FP64 divisions, so one wave of the iteration before evaluates them
// and the others read them with their clock: a launch of 556 x 701 in FP64 with
// rain, evaporation and two sources 30.3 -> 27.0 us, of 256^2 with rain 14.0 ->
// 13.3.  With an adaptive step the length of the iteration is not known yet:
// those waves evaluate the rates at t + dt themselves.
__device__ __forceinline__ void note_forcing(const StepCommon &s, int slot, double t, int lane)
{
    const double tm = t + s.dt_fixed;
    if (lane < 4) {
        // rain_rate and evap_rate, side by side
        const bool ev = lane & 2, on = ev ? s.evap_on : s.nrain > 0;
        double r = 0.0;
        if (on)
            r = series_value(ev ? s.evapo : s.rain, ev ? s.nevapo : s.nrain, s.dtrain, (lane & 1) ? tm : t) /
                (s.dtrain * 1000.0);
        s.clk[slot].force[lane] = r;
    }
    for (int i = lane; i < 2 * s.nst; i += 64)
        s.src_rate[(size_t)slot * 2 * s.nst + i] = source_rate(s, i >> 1, (i & 1) ? tm : t);
}

template <typename F>
__device__ void bookkeeping(const StepCommon &s, const Iter &it, const StepTime &st, const F &vel,
                            const int part, const int lane, const bool forcing)
{
    if (part >= kBookParts) {
        const int i = (part - kBookParts) * 64 + lane;
        if (i < s.nbc) {
            const int r = s.bc_r[i], j = s.bc_c[i];
            double hh, ua, va;
            vel(r, j, hh, ua, va);
            s.bc_acc[i] += bc_rate(s.bc_kind[i], hh, ua, va, s.dx, s.dy) * st.dt2;
        }
        return;
    }
    if (part == 0) {
        const double tn = st.tm + st.dt;
        if (lane == 0) {
            Clock &nb = s.clk[it.slot_b];
            nb.t = tn;
            nb.dt2_prev = st.dt2;
            nb.mstep = s.clk[it.slot_a].mstep + 2;
        }
        if (lane < kCflSlots) s.clk[it.slot_c].cfl[lane].bits = kInfBits;
        if (forcing) note_forcing(s, it.slot_b, tn, lane);
        return;
    }
    if (it.step_index > 0) {
        double vol, src, clip, qo;
        reduce_partials(it.part_in, s.nparts, lane, vol, src, clip, qo);
        if (lane == 0) {
            Ledger &L = *s.ledger;
            double dt2p = s.clk[it.slot_a].dt2_prev;
            L.v_src += src * s.dx * s.dy;
            L.v_clip += clip * s.dx * s.dy;
            L.v_out += qo * dt2p;
            L.q_last = qo;
            if (qo > L.q_peak) { L.q_peak = qo; L.t_peak = st.t; }
            L.vol_last = vol * s.dx * s.dy;
            L.reduced += 1;
            long long i = it.step_index - 1;
            if (s.hydro && i < s.hydro_cap) {
                s.hydro[2 * i] = st.t;
                s.hydro[2 * i + 1] = qo;
            }
        }
    }
}

// Ledger view for the host: the committed ledger plus the partials of the
// last iteration, which the next iteration would reduce.
__device__ __forceinline__ void ledger_peek(const StepCommon &s, Ledger *out, const int lane)
{
    const Iter it = iter_of(s);
    double vol = 0, src = 0, clip = 0, qo = 0;
    if (it.step_index > 0) reduce_partials(it.part_in, s.nparts, lane, vol, src, clip, qo);
    if (lane == 0) {
        Ledger L = *s.ledger;
        if (it.step_index > 0) {
            double dt2p = s.clk[it.slot_a].dt2_prev;
            double t = s.clk[it.slot_a].t;
            L.v_src += src * s.dx * s.dy;
            L.v_clip += clip * s.dx * s.dy;
            L.v_out += qo * dt2p;
            L.q_last = qo;
            if (qo > L.q_peak) { L.q_peak = qo; L.t_peak = t; }
            L.vol_last = vol * s.dx * s.dy;
            L.reduced += 1;
            long long i = it.step_index - 1;
            if (s.hydro && i < s.hydro_cap) {
                s.hydro[2 * i] = t;
                s.hydro[2 * i + 1] = qo;
            }
        }
        *out = L;
    }
}

}  // namespace sw2d
