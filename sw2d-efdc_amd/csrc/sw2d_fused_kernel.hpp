// sw2d_fused_kernel.hpp -- one fused kernel per SW2D loop iteration.
//
// The reference (SW2D-EFDC.cu:4798-4877) runs nine grid-stride kernels per
// iteration over ~20 FP64 arrays: flux, continuity, treat_error, continuity,
// hm_hn, uu1_vv1, uu_vv, uua_vva, forward.  The complete state between
// iterations is only (h, um, vn) (bed z is constant); every other array is a
// local function of it.  This kernel reads (h, um, vn, z) once and writes
// (h, um, vn) once per iteration: 56 B/cell in FP64; 32 B/cell in the FP32
// form, whose bed is not rounded to binary32 (it is input data: rounding a
// DEM to binary32 moves it by up to half an ulp of its relief, which alone
// shifts depths by ~1 mm on a 2.5 m-relief test DEM, while FP32 state costs
// 0.2 mm): it reads, in the same 8 bytes, the cell's bed steps to its north
// and west neighbours, the FP64 differences rounded once at creation.
//
// Work decomposition.  A tile is one wavefront (64 lanes) and covers 58
// output columns x H output rows.  Lane l holds column j = j0 - 3 + l: the
// dependency chain flux(+-1) -> continuity (+-1) -> treat_error (+-1) ->
// continuity needs 3 cells of halo on each side.  The wave streams the rows
// of its tile from north to south; when row k arrives it computes
//   the face depths/velocities of row k            (hm_hn, uu1_vv1, uua_vva)
//   the fluxes of row k-1                          (flux)
//   the first continuity of row k-2                (continuity at t)
//   treat_error on the faces of row k-2
//   the second continuity of row k-3              (continuity at t + dt)
// and stores row k-3 of the new state.  Values of a row are carried in
// registers while they are needed; east/west neighbours are DPP lane moves,
// made afresh in the row that uses them rather than carried to the next one:
// register pressure sets the waves per SIMD.  No LDS staging and no
// barriers: each wave is independent.  The grid is one wave per tile plus the
// bookkeeping waves.
//
// What bounds it: the number of instructions, scalar ones as much as vector ones
// (a wave issues one in 4 to 5 cycles whatever its dependencies, and the waves of
// a SIMD get in each other's way), and on states past the 256 MB cache the loads
// in flight.  So the row is written for few instructions: the conditions are lane
// masks on the scalar unit, each upwind product is formed once (the south one of a
// row is the north one of the next, the east one of a cell the west one of its
// east neighbour), the weirs, the momentum update and the first continuity run
// only in rows where a lane needs them, a row without fluxes and sources keeps its
// depths, what changes only at the first or last rows of a tile (rows outside the
// grid, rows before the first output) is set there and not tested in every row,
// and the three rows above a tile run in a short loop of their own.  Measured per
// launch against per-row tests, selects and resources, and with the FP64 power's
// coefficients from LDS, same results: one 2048^2 grid FP32 57.8 -> 51.2 us, FP64
// 127 -> 118; 1537 x 2311 mixed 54.5 -> 47.2; 331 x 1009 FP32 17.5 -> 16.1; 256^2
// FP64 13.2 -> 12.1; 24 grids of 128^2..1024^2 FP64 158 -> 144.
//
// T is the type of the fluxes and of the momentum arithmetic, TH that of the
// depths, the continuity updates and every switch that tests a depth.
// Instantiated three times: sw2d_fused64.hip (T = TH = double, built with
// -ffp-contract=off: every FP64 expression is written in the reference's
// evaluation order, so the results equal the reference arithmetic as restated
// by the CPU FP64 check, bit for bit), sw2d_fused32.hip (T = TH = float) and
// sw2d_fusedmix.hip (T = float, TH = double: FP32 fluxes and momentum
// arithmetic over FP64 depths, so the dry-bed and threshold switches see the
// depths the FP64 form sees).
#pragma once
#include "sw2d_common.hpp"

namespace sw2d {

// Wave-wide predicates are kept as 64-bit lane masks in scalar registers: a
// comparison writes one directly, the logic between them (which face is
// active, which of the flux's branches applies, the west neighbour's bit) runs
// on the scalar unit, and lanes() turns a mask back into the per-lane
// condition of a select at no cost.  Per-lane booleans carried from row to row
// or across a branch cost two vector instructions at every vote (0/1 and back).
typedef unsigned long long u64;
__device__ __forceinline__ u64 vote(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ bool lanes(u64 m) { return __builtin_amdgcn_inverse_ballot_w64(m); }

// 1 for a mask with a lane in it, else 0, on the scalar unit
__device__ __forceinline__ unsigned any_lane(u64 m)
{
    unsigned n;
    asm("s_bcnt1_i32_b64 %0, %1" : "=s"(n) : "s"(m) : "scc");
    return n < 1u ? n : 1u;
}
// keeps a rarely taken branch one: the compiler would make selects of it, which
// every row would execute
__device__ __forceinline__ void keep_branch() { asm volatile(""); }
// One scenario array, read and written through a buffer resource (base and
// range in scalar registers): a lane's byte offset within the row stays in one
// register for the whole tile and the row's byte offset is scalar, so a row
// costs no address arithmetic on the vector unit.  Offsets stay below 2^32
// (cells below 2^29, which the host enforces).  A lane outside the grid or the
// tile's output columns has the offset kOutside, past the range of any array:
// its loads return 0, which is the ghost value, and its stores are dropped.
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
constexpr unsigned kOutside = 0xffffff80u;
template <typename V> struct Arr {
    void *p;
    unsigned bytes;
    __device__ Arr(const void *q, unsigned cells)
        : p(const_cast<void *>(q)), bytes(cells * (unsigned)sizeof(V)) {}
    // 0x00020000: the 32-bit data format (a buffer with the invalid format reads
    // zeros)
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc() const
    {
        return __builtin_amdgcn_make_buffer_rsrc(p, (short)0, bytes, 0x00020000);
    }
    __device__ __forceinline__ V load(unsigned off, unsigned row) const
    {
        const unsigned ro = row * (unsigned)sizeof(V);
        if constexpr (sizeof(V) == 1)
            return __builtin_amdgcn_raw_buffer_load_b8(rsrc(), (int)off, (int)ro, 0);
        else if constexpr (sizeof(V) == 4)
            return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(rsrc(), (int)off, (int)ro, 0));
        else
            return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(rsrc(), (int)off, (int)ro, 0));
    }
    __device__ __forceinline__ void store(unsigned off, unsigned row, V v) const
    {
        const unsigned ro = row * (unsigned)sizeof(V);
        if constexpr (sizeof(V) == 4)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rsrc(), (int)off, (int)ro, 0);
        else
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rsrc(), (int)off, (int)ro, 0);
    }
};

// New flux of a face between a cell ("o") and its north or west neighbour
// ("b"), SW2D-EFDC.cu:97-353: the dry-bed weirs B1 (surface below the
// neighbour's bed), B2 (the neighbour's below this bed) and B3 (one side dry)
// all read (coef * hv) * sqrt(c2 * hv), every other face the momentum update
// B4.  act: the faces to update (0 elsewhere); Wo, Wb: the sides' depths above
// th; Lo, Lb: below it, so B3's "(h_o - th)(h_b - th) < 0" is mask logic.
// mom(face depth, its B4 faces, surface difference, friction faces) gives B4.
// FP32 depths test the water surfaces through the bed step dz = z_b - z_o,
// FP64 ones through the elevations.
template <typename T, typename TH, typename Mom>
__device__ __forceinline__ T face_flux(const u64 act, const TH ho, const TH hb, const T dz,
                                       const double zo, const double zb, const u64 Wo,
                                       const u64 Wb, const u64 Lo, const u64 Lb, const TH thh,
                                       const T gg, const Mom &mom)
{
    using M = num<T>;
    constexpr bool kH32 = sizeof(TH) == 4;
    u64 B1, B2;
    double eo = 0, eb = 0;
    if constexpr (kH32) {
        B1 = vote(ho < dz);
        B2 = vote(hb < -dz) & ~B1;
    } else {
        eo = ho + zo;
        eb = hb + zb;
        B1 = vote(eo < zb);
        B2 = vote(eb < zo) & ~B1;
    }
    const u64 B3 = ((Wo & Lb) | (Lo & Wb)) & ~(B1 | B2);
    const u64 weir = act & (B1 | B2 | B3), B4 = act & ~weir;
    T val = 0;
    if (weir) {
        T coef = T(0.5440), hv = lanes(B2) ? (T)ho : (T)hb, c2 = gg;
        if (B3 & act) {
            T hv3;  // max(surfaces) - max(beds)
            if constexpr (kH32)
                hv3 = (dz <= T(0)) ? M::max_(ho, hb + dz) : M::max_(ho - dz, hb);
            else
                hv3 = (T)(__builtin_fmax(eo, eb) - __builtin_fmax(zo, zb));
            coef = lanes(B3) ? T(0.350) : coef;
            hv = lanes(B3) ? hv3 : hv;
            c2 = lanes(B3) ? T(2.00) * gg : c2;
        }
        const T w = coef * hv * M::sqrt_(c2 * hv);
        const u64 back = B2 | (B3 & Wo);  // flow toward the neighbour
        const u64 wet = (B1 & Wb) | (B2 & Wo) | B3;
        val = lanes(back) ? -w : w;
        val = lanes(weir & wet) ? val : T(0);
    }
    if (B4) {
        const TH hfd = TH(0.50) * (ho + hb);
        T dsurf;
        if constexpr (kH32) dsurf = (ho - hb) - dz;
        else dsurf = (T)(eo - hb - zb);
        const T up = mom((T)hfd, dsurf, B4 & vote(!(hfd <= thh)));
        val = lanes(B4) ? up : val;
    }
    return val;
}

// the tables of the power, to be read anew at each use
template <typename T>
__device__ __forceinline__ PowTablesLds pow_tables(const double *t)
{
    if constexpr (sizeof(T) == 4) return PowTablesLds{t, 0};
    int zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    return PowTablesLds{t, zero};
}

constexpr int kMaxTileRows = 512;

// Waves per SIMD that the registers have to leave room for.  Each of them issues
// about one instruction in 4 to 5 cycles, so SIMDs are filled by more of them: a
// row takes a wave (2.0 + w) units of time beside w - 1 others in the FP32 and
// mixed forms, (0.8 + w) in FP64 (2048^2 and 331 x 1009 grids at w = 1 to 5).
// 3 against 2 in FP64: 2048^2 134 -> 125 us when it came; 4 (128 registers) spill:
// 107 -> 137.  5 against 4 in FP32: 2048^2 59.0 -> 56.8 when it came; 6 (80
// registers) spill in the storm's instantiation: 50.4 -> 53.1.
template <typename T>
constexpr int kMinWaves = (sizeof(T) == 8 ? 3 : 5);

// F: the features (kFeat*) this instantiation handles.  A feature missing
// from F is compiled out (its uniforms, branches and loops), which the host
// may only do for launches where no scenario uses it.  The arithmetic of
// what remains is the same in every instantiation (FP64 fuses no
// multiply-add, FP32 only within one source expression), so a scenario's
// results do not depend on the instantiation that ran it.
template <typename T, typename TH, int F>
__global__ void __launch_bounds__(64, (kMinWaves<T>))
fused_step(const Scenario *__restrict__ scen, const TileRef *__restrict__ tiles, const int nblocks,
           const int phase)
{
    using M = num<T>;
    using MH = num<TH>;
    constexpr bool kStorm = F & kFeatStorm, kSources = F & kFeatSources;
    constexpr bool kAdaptive = F & kFeatAdaptive, kMap = F & kFeatMap;
    const int lane = threadIdx.x;

    // block -> (scenario, block within it).  The hardware deals consecutive
    // blocks to the 8 XCDs in turn; the remap gives each XCD runs of kRun blocks
    // of the block list, so that neighbouring tiles share an L2, and the XCDs
    // share what is wet: with one run an XCD, the XCD of a lake or a wave front
    // ended last (4096^2 in FP32 148 -> 142 us, 556 x 701 FP64 25.1 -> 23.4,
    // 2048^2 FP64 118 -> 114; runs of 4 and 16 blocks share less: 151 and 144).
    int b = blockIdx.x;
    {
        constexpr int kXcd = 8, kRun = 128;
        const int base = b / (kXcd * kRun) * (kXcd * kRun), left = nblocks - base;
        const int i = b - base, x = i % kXcd, per = left / kXcd, rem = left % kXcd;
        b = base + i / kXcd + (left >= kXcd * kRun ? x * kRun : x * per + (x < rem ? x : rem));
    }
    int sid = 0, local = b;
    if (tiles) {
        const TileRef t = tiles[b];
        sid = t.sid;
        local = t.local;
    }
    // the descriptor is read in place (no local copy: its uniform fields stay
    // reloadable scalar loads instead of pinned registers)
    const Scenario &d = scen[sid];
    const StepCommon &s = d.s;
    // iteration k of this scenario: k mod 6 from the launch phase, k itself
    // from the clock slot the previous iteration wrote
    const int k6 = (phase - d.phase0 + 6) % 6;
    Iter it;
    it.slot_a = k6 % 3; it.slot_b = (k6 + 1) % 3; it.slot_c = (k6 + 2) % 3;
    it.part_out = d.part + (size_t)(k6 & 1) * s.nparts;
    it.part_in = d.part + (size_t)((k6 + 1) & 1) * s.nparts;
    it.step_index = s.clk[it.slot_a].mstep >> 1;
    const StepTime st = step_time<kAdaptive>(s, it);
    if (d.status) {
        // batch member: a finished scenario leaves its blocks idle
        if (d.status->done) return;
        if (!(it.step_index < d.k_end && st.t + st.dt <= d.t_end)) {
            if (local == 0 && lane == 0) d.status->done = 1;
            return;
        }
    }
    const int ib = k6 & 1;
    // the bookkeeping waves come first, so that the reduction of the last
    // iteration's partial sums runs beside the tiles and not after them
    const int nbook = d.nblocks - d.ntiles;
    const int tile = local < nbook ? d.ntiles + local : local - nbook;
    if (tile >= d.ntiles) {
        PitchedState<T, TH> ps{(const TH *)d.st[ib][0], (const T *)d.st[ib][1],
                               (const T *)d.st[ib][2], s.R, s.C, d.P, (TH)s.th};
        auto vel = [&](int r, int j, double &hh, double &ua, double &va) {
            hh = (double)ps.hv(r, j);
            ua = (double)ps.uua(r, j);
            va = (double)ps.vva(r, j);
        };
        const int part = local;
        bookkeeping(s, it, st, vel, part, lane, true);
        if (part == 0 && lane == 0 && d.status) {
            const long long kn = it.step_index + 1;
            const double tn = st.tm + st.dt;
            d.status->k = kn;
            d.status->t = tn;
            // the flag the kernel reads (done) is only set by a later launch;
            // fin tells the host now that nothing more will run
            if (kn >= d.k_end || (s.fixed_dt && !(tn + s.dt_fixed <= d.t_end))) d.status->fin = 1;
        }
        return;
    }

    const int strip = tile % d.nstrips, chunk = tile / d.nstrips;
    const int R = s.R, C = s.C, P = d.P;
    const int j0 = strip * d.W;
    const int j = j0 - 3 + lane;
    const bool colout = (lane >= 3) && (lane < 3 + d.W) && (j < C);
    const u64 out_cols = vote(colout);
    const int r0 = chunk * d.H;
    const int r1 = (r0 + d.H < R) ? r0 + d.H : R;

    // software pipeline: row k+1 is loaded while row k is processed; the first
    // row's loads are issued before the forcing is evaluated.  Rows and columns
    // outside the grid read the ghost values 0 and are inactive.
    const unsigned cells = (unsigned)R * (unsigned)P;
    const Arr<TH> h_in(d.st[ib][0], cells), h_out(d.st[ib ^ 1][0], cells);
    const Arr<T> um_in(d.st[ib][1], cells), um_out(d.st[ib ^ 1][1], cells);
    const Arr<T> vn_in(d.st[ib][2], cells), vn_out(d.st[ib ^ 1][2], cells);
    // FP32 arithmetic: storm factors and source terms in FP32.  FP32 depths:
    // water-surface tests from bed differences carried per face (z stays
    // FP64 only to form them) and stochastically rounded depth updates.
    constexpr bool kF32 = sizeof(T) == 4;
    constexpr bool kH32 = sizeof(TH) == 4;
    // the bed: FP64 elevations, or in the FP32 form the cell's bed-step pair
    // (8 bytes as well; read as one double's bits); NaN marks an inactive cell
    const Arr<const double> zg(kH32 ? d.dz : d.z, cells);
    const bool map_on = kMap && s.ncls_on;
    const Arr<uint8_t> cls_in(map_on ? (const void *)d.cls : (const void *)d.z, map_on ? cells : 0u);
    // Manning coefficients of the classes; without a map every cell reads class
    // 0 (an empty array), which is the scenario's coefficient
    __shared__ T nt_s[kMaxClasses];
    if (kMap && lane < kMaxClasses) nt_s[lane] = (T)(map_on ? s.ntab[lane] : s.rn);
    // FP64: the tables of the power in LDS.  Reads of them from memory share the
    // counter of the row loads, and waiting for one of the former waits for the
    // next row as well: four such waits a row with friction on both faces.  24
    // grids of 128^2..1024^2 221 -> 195 us a launch, one of 2048^2 140 -> 134.
    __shared__ double pow_s[kF32 ? 2 : kPowLds];
    if constexpr (!kF32) {
        pow_s[lane] = kPowRecip[lane];
        pow_s[64 + lane] = kPowNlog[lane];
        pow_s[128 + lane] = kPowExp2[lane];
        if (lane < 16) pow_s[192 + lane] = kPowCoefMem[lane];
    }
    // lanes read what others wrote (the block is one wave: this orders, it does
    // not wait)
    if constexpr (kMap || !kF32) __syncthreads();
    const int kbeg = r0 - 3, kend = r1 + 3, kload = kend < R ? kend : R;
    // Row to load next: its offset (in elements), and the lanes' byte offsets.
    // While that row is outside the grid (or past the last one that is needed)
    // every lane's offset is kOutside, so it reads ghosts; a branch around the
    // loads would make the count of accesses in flight unknown, and the next
    // row's wait would cover the prefetched row as well.  aim() sets them for
    // row k; it is called where they change (row kaim) and nowhere else.
    unsigned offT, offH, off8, off1, row_in = 0, row_step;
    u64 cols_n;  // lanes inside the grid in that row
    int kaim;
    auto aim = [&](const int k) {
        const bool on = k >= 0 && k < kload;
        int c = j;
        asm volatile("" : "+v"(c));  // computed here: not held in registers
        const bool in = on && c >= 0 && c < C;
        offT = in ? (unsigned)c * (unsigned)sizeof(T) : kOutside;
        offH = in ? (unsigned)c * (unsigned)sizeof(TH) : kOutside;
        off8 = in ? (unsigned)c * 8u : kOutside;
        off1 = in ? (unsigned)c : kOutside;
        cols_n = vote(in);
        row_in = on ? (unsigned)k * (unsigned)P : 0u;
        row_step = on ? (unsigned)P : 0u;
        kaim = k < 0 ? 0 : k < kload ? kload : 0x7fffffff;
    };
    TH nh;
    T nu, nv;
    double nz;
    uint8_t ncl;
    auto load_row = [&]() {
        nh = h_in.load(offH, row_in);
        nu = um_in.load(offT, row_in);
        nv = vn_in.load(offT, row_in);
        nz = zg.load(off8, row_in);
        if constexpr (kMap) ncl = cls_in.load(off1, row_in);
        else ncl = 0;
    };
    aim(kbeg);
    load_row();

    // CFL candidates only for an adaptive time step; a wave-uniform flag, so
    // a scenario runs the same instructions alone and in a mixed batch
    const bool adapt = kAdaptive && !s.fixed_dt;
    const bool storm_on = kStorm && s.storm_on;
    // the scenario's point sources, where one lies among the tile's columns and
    // the rows of its first continuity
    int nst = kSources ? s.nst : 0;
    if (nst > 0) {
        bool here = false;
        for (int i = lane; i < nst; i += 64) {
            const int r = s.src_r[i], c = s.src_c[i] - (j0 - 3);
            here |= r >= r0 - 1 && r <= r1 && c >= 0 && c < 64;
        }
        if (!vote(here)) nst = 0;
    }
    const double *src_rate = s.src_rate + (size_t)it.slot_a * 2 * s.nst;
    const T gg = (T)s.g, dx = (T)s.dx;  // cells are square: dy = dx
    const TH thh = (TH)s.th;
    const T rdx = (T)(1.0 / s.dx);
    const T dt2 = (T)st.dt2;
    const TH dt2h = (TH)st.dt2;
    const T dt2dx = (T)(st.dt2 / s.dx);
    // FP32 momentum: the upwind differences carry sums of two face
    // velocities, so dt2/dx enters with the two halvings folded
    const T dt2dx4 = T(0.25) * dt2dx, dt2half = T(0.5) * dt2;
    const T rn = (T)s.rn;

    // forcing of this iteration: first continuity at t, second at t + dt
    // (note_forcing)
    const Clock &ck = s.clk[it.slot_a];
    const double rr1 = ck.force[0], ev1 = ck.force[2];
    const double rr2 = adapt ? rain_rate(s, st.tm) : ck.force[1];
    const double ev2 = adapt ? evap_rate(s, st.tm) : ck.force[3];
    const bool storm1 = storm_live(s, st.t), storm2 = storm_live(s, st.tm);
    double gx1 = 0, gx2 = 0;
    T pk1 = 0, pk2 = 0;  // FP32 form: peak * gx of this column, 0 outside the storm window
    __shared__ T gy_s[2][kMaxTileRows + 8];
    if (storm_on) {
        const double x = ((double)j + 0.5) * s.dx;
        gx1 = storm_factor(x - (s.st_x0 + s.st_vx * st.t), s.st_sigma);
        gx2 = storm_factor(x - (s.st_x0 + s.st_vx * st.tm), s.st_sigma);
        pk1 = storm1 ? (T)(s.st_peak * gx1) : T(0);
        pk2 = storm2 ? (T)(s.st_peak * gx2) : T(0);
        for (int i = lane; i < d.H + 6; i += 64) {
            const double y1 = ((double)(r0 - 5 + i) + 0.5) * s.dy;
            const double y2 = ((double)(r0 - 6 + i) + 0.5) * s.dy;
            gy_s[0][i] = (T)storm_factor(y1 - (s.st_y0 + s.st_vy * st.t), s.st_sigma);
            gy_s[1][i] = (T)storm_factor(y2 - (s.st_y0 + s.st_vy * st.tm), s.st_sigma);
        }
        __syncthreads();
    }
    const T rr1t = (T)rr1, rr2t = (T)rr2, ev1t = (T)ev1, ev2t = (T)ev2;
    const T P_lake = (T)s.P_lake, P_land = (T)s.P_land;
    const TH ewl = (TH)s.EV_WL_min;
    // no water is added or taken in the second continuity: a row without
    // fluxes then keeps its depths
    const bool calm2 = !storm_on && nst == 0 && rr2 == 0.0 && ev2 == 0.0;
    // one forcing for all depths (no evaporation, the same fraction of the rain)
    const bool even = s.P_lake == s.P_land && ev1 == 0.0 && ev2 == 0.0;
    // the scenario's conditions as bits of one register, tested where they are
    // needed (as conditions they take two registers each, too many to keep)
    enum : unsigned { kOnStorm = 1, kOnStorm1 = 2, kOnStorm2 = 4, kOnCalm = 8, kOnEven = 16 };
    const unsigned on_bits = (unsigned)__builtin_amdgcn_readfirstlane(
        (storm_on ? kOnStorm : 0u) | (storm1 ? kOnStorm1 : 0u) | (storm2 ? kOnStorm2 : 0u) |
        (calm2 ? kOnCalm : 0u) | (even ? kOnEven : 0u));
    const int out_edge = __builtin_amdgcn_readfirstlane(s.out_edge);

    // the outlet's row, where its column is among this wave's lanes, and its lane
    const int ol = s.out_edge ? s.out_c - (j0 - 3) : -1;
    const int orow = (ol >= 0 && ol < 64) ? s.out_r : -1000;
    const u64 out_lane = 1ull << (ol & 63);
    T qo_eff = 0;

    // carried rows: suffix 1 = row k-1, 2 = k-2, 3 = k-3.  Masks: A active,
    // W deeper than th, L shallower
    TH h1 = 0, h2 = 0, h3 = 0;
    double z1 = 0, z2 = 0;
    u64 A1 = 0, A2 = 0, A3 = 0, W1 = 0, W2 = 0, L1 = 0, L2 = 0;
    T u1 = 0, v1 = 0;
    T uu1_1 = 0, vv1_1 = 0, vv1_2 = 0;
    T px1 = 0, py1 = 0;    // upwind products between rows k-2 and k-1
    T dzn1 = 0, dzw1 = 0;  // FP32 form: z(k-2) - z(k-1) and z(k-1, j-1) - z(k-1, j)
    T nc1 = rn, nc2 = rn;
    T umnP = 0, vnnP = 0, umpP = 0, vnpP = 0;
    // rows with faces that may carry flux: bit 0 north faces, bit 1 west faces of
    // row k-1, bits 2 and 3 of row k-2, and so on
    unsigned flow = 0;
    unsigned outT = kOutside, outH = kOutside, row_out = 0;  // of the next row to store
    const int kcfl = adapt ? r1 : -1000;
    u64 D1 = 0;  // cells of row k-3 that dried in the first continuity
    T div1 = 0;  // its flux divergence of row k-3, and which fluxes of it were taken out
    unsigned cut1 = 0;

    // sums over all lanes; those outside the output columns are dropped at the end
    // (the clipped volume, which few rows add to, in LDS)
    double acc_vol = 0, acc_src = 0;
    __shared__ double clip_s[64];
    clip_s[lane] = 0.0;
    // CFL: the largest |u| + sqrt(g h) of either direction; min_f dx / s_f =
    // dx / max_f s_f because rounding dx / s is monotone in s (and dy = dx)
    T smax = 0;

    // row k: what the rows after it need of it
    struct Front {
        TH h, hm, hn;
        T u, v, uu1, uu1w, vv1, px, py, dzn, dzw, nc;
        double z;
        u64 A, W, L;
    };
    auto front = [&](const int k) __attribute__((always_inline)) -> Front {
        Front o;
        o.h = nh; o.u = nu; o.v = nv; o.z = nz;
        const uint8_t cl = ncl;
        const u64 cols = cols_n;
        row_in += row_step;
        if (k + 1 == kaim) aim(k + 1);
        load_row();
        // FP32 form: z holds the bed steps of row k's cell to its north (low
        // word) and west (high word) neighbours, NaN for an inactive cell
        const u32x2 zsteps = __builtin_bit_cast(u32x2, o.z);
        o.dzn = (T)__uint_as_float(zsteps.x);
        o.dzw = (T)__uint_as_float(zsteps.y);
        o.A = vote(kH32 ? (o.dzw == o.dzw) : (o.z == o.z)) & cols;
        o.W = vote(o.h > thh);
        o.L = vote(o.h < thh);
        o.nc = rn;
        if constexpr (kMap) o.nc = nt_s[cl];

        // ---- face depths and velocities (hm_hn, uu1_vv1) ----
        // (row 0's north and column 0's west faces carry no flux, so their
        // velocities are 0 whatever the face depth)
        o.hn = TH(0.50) * (o.h + from_west(o.h));
        o.hm = TH(0.50) * (o.h + h1);
        o.uu1 = (o.hm >= thh) ? M::div_(o.u, (T)o.hm) : T(0.00);
        o.vv1 = (o.hn >= thh) ? M::div_(o.v, (T)o.hn) : T(0.0);

        // upwind products of the convection terms between rows k-1 and k: the
        // south one of row k-1 and the north one of row k, so each is formed
        // once and carried.  FP32: without the halvings (see dt2dx4)
        o.uu1w = from_west(o.uu1);
        if constexpr (kF32) {
            const T sr = o.uu1 + uu1_1;
            o.px = sr * (o.u + u1) + M::abs_(sr) * (u1 - o.u);
            const T sa = o.uu1 + o.uu1w;
            o.py = sa * (o.v + v1) + M::abs_(sa) * (v1 - o.v);
        } else {
            const T ur = T(0.50) * (o.uu1 + uu1_1);
            o.px = ur * (o.u + u1) * T(0.50) + M::abs_(ur) * (u1 - o.u) * T(0.50);
            const T av = T(0.50) * (o.uu1 + o.uu1w);
            o.py = av * (o.v + v1) * T(0.50) + M::abs_(av) * (v1 - o.v) * T(0.50);
        }
        return o;
    };
    auto push = [&](const Front &o) __attribute__((always_inline)) {
        h3 = h2; h2 = h1; h1 = o.h;
        z2 = z1; z1 = o.z;
        A3 = A2; A2 = A1; A1 = o.A;
        W2 = W1; W1 = o.W;
        L2 = L1; L1 = o.L;
        u1 = o.u; v1 = o.v;
        uu1_1 = o.uu1;
        vv1_2 = vv1_1; vv1_1 = o.vv1;
        px1 = o.px; py1 = o.py;
        dzn1 = o.dzn; dzw1 = o.dzw;
        nc2 = nc1; nc1 = o.nc;
    };

    // the three rows above feed the window only
    for (int k = kbeg; k < r0; ++k) push(front(k));
    // everything loaded so far is here (vmcnt, lgkmcnt 0): the loop's own waits
    // then count only its own accesses (a wait for a load from before it would
    // be a wait for the stores of the row before in every later row)
    __builtin_amdgcn_s_waitcnt(0x0070);
    for (int k = r0; k < kend; ++k) {
        unsigned on = on_bits;
        asm volatile("" : "+s"(on));
        const Front o = front(k);
        const TH hm0d = o.hm, hn0d = o.hn;
        const T hm0 = (T)hm0d, hn0 = (T)hn0d, uu1_0 = o.uu1, vv1_0 = o.vv1, px0 = o.px, py0 = o.py;
        const T uu1_0w = o.uu1w;
        const u64 A0 = o.A;

        if (k < kcfl) {
            // CFL candidates of the incoming state on the faces of row k
            if (lanes(A0 & A1 & out_cols & vote(hm0d > thh))) {
                const T w = M::abs_(uu1_0) + M::sqrt_(gg * hm0);
                smax = (w > smax) ? w : smax;
            }
            if (lanes(A0 & (A0 << 1) & out_cols & vote(hn0d > thh))) {
                const T w = M::abs_(vv1_0) + M::sqrt_(gg * hn0);
                smax = (w > smax) ? w : smax;
            }
        }

        // ---- fluxes of row f = k-1 (flux, SW2D-EFDC.cu:97-353) ----
        const int f = k - 1;
        T umn = 0, vnn = 0;
        // x direction: um at the north face of (f, j); w = row f-1, e = row f
        // y direction: vn at the west face of (f, j); s = column j-1, n = column j
        const u64 FX = A1 & A2 & (W1 | W2);
        const u64 FY = A1 & (A1 << 1) & (W1 | (W1 << 1));
        flow <<= 2;
        if (FX) {
            flow |= 1u;
            umn = face_flux<T, TH>(FX, h1, h2, dzn1, z1, z2, W1, W2, L1, L2, thh, gg,
                                   [&](const T hm1, const T dsurf, const u64 fr) {
                const T u13 = gg * hm1 * dt2dx * dsurf;
                // the upwind product across the cell's west side; its east
                // side's is the east neighbour's
                const T u1w = from_west(u1);
                T u11, u12, pd;
                if constexpr (kF32) {
                    const T sd = vv1_1 + vv1_2;
                    pd = sd * (u1w + u1) + M::abs_(sd) * (u1w - u1);
                    u11 = dt2dx4 * (px0 - px1);
                    u12 = dt2dx4 * (from_east(pd) - pd);
                } else {
                    const T vd = T(0.50) * (vv1_1 + vv1_2);
                    pd = vd * (u1w + u1) * T(0.50) + M::abs_(vd) * (u1w - u1) * T(0.50);
                    u11 = dt2dx * (px0 - px1);
                    u12 = dt2dx * (from_east(pd) - pd);
                }
                u12 = (j != 0) ? u12 : T(0);
                // uua_vva (489-522): vva of row f
                const T vva1 = T(0.250) * (vv1_1 + from_east(vv1_1) + vv1_2 + from_east(vv1_2));
                const T nf = kMap ? T(0.5) * (nc2 + nc1) : rn;  // rn itself without a map
                T ram = 0.00;
                if (lanes(fr)) {
                    const T sqx = M::sqrt_(uu1_1 * uu1_1 + vva1 * vva1);
                    ram = M::div_(gg * nf * nf * sqx, pow1333(hm1, pow_tables<T>(pow_s)));
                }
                if constexpr (kF32) {
                    const T a = dt2half * ram;
                    return M::div_((T(1.00) - a) * u1 + (-u11 - u12 - u13), T(1.00) + a);
                } else {
                    return M::div_((T(1.00) - dt2 * ram * T(0.50)) * u1 + (-u11 - u12 - u13),
                                   T(1.00) + dt2 * ram * T(0.50));
                }
            });
        }
        if (FY && k < r1 + 2) {
            flow |= 2u;
            vnn = face_flux<T, TH>(FY, h1, from_west(h1), dzw1, z1, kH32 ? 0.0 : from_west(z1), W1,
                                   W1 << 1, L1, L1 << 1, thh, gg,
                                   [&](const T hn1, const T dsurf, const u64 fr) {
                const T v13 = gg * hn1 * dt2dx * dsurf;
                const T v1w = from_west(v1), uu1_1w = from_west(uu1_1);
                T v11, v12, pd;
                if constexpr (kF32) {
                    const T sq = vv1_1 + from_west(vv1_1);
                    pd = sq * (v1w + v1) + M::abs_(sq) * (v1w - v1);
                    v11 = dt2dx4 * (py0 - py1);
                    v12 = dt2dx4 * (from_east(pd) - pd);
                } else {
                    const T qv = T(0.50) * (vv1_1 + from_west(vv1_1));
                    pd = qv * (v1w + v1) * T(0.50) + M::abs_(qv) * (v1w - v1) * T(0.50);
                    v11 = dt2dx * (py0 - py1);
                    v12 = dt2dx * (from_east(pd) - pd);
                }
                v11 = (f != 0) ? v11 : T(0);
                // uua_vva (489-522): uua of row f
                const T uua1 = T(0.250) * (uu1_1 + uu1_0 + uu1_1w + uu1_0w);
                const T nf = kMap ? T(0.5) * (from_west(nc1) + nc1) : rn;
                T ram = 0.00;
                if (lanes(fr)) {
                    const T sqy = M::sqrt_(uua1 * uua1 + vv1_1 * vv1_1);
                    ram = M::div_(gg * nf * nf * sqy, pow1333(hn1, pow_tables<T>(pow_s)));
                }
                if constexpr (kF32) {
                    const T a = dt2half * ram;
                    return M::div_((T(1.00) - a) * v1 + (-v11 - v12 - v13), T(1.00) + a);
                } else {
                    return M::div_((T(1.00) - dt2 * ram * T(0.50)) * v1 + (-v11 - v12 - v13),
                                   T(1.00) + dt2 * ram * T(0.50));
                }
            });
        }

        // ---- first continuity of row g = k-2 at time t (602-664) ----
        // it only decides which cells dry, so rows whose faces (their own and
        // the next row's north ones) carry nothing skip it
        const int g = k - 2;
        u64 D0 = 0;
        T umpg = umnP, vnpg = vnnP, div0 = 0;
        unsigned cut = 0;  // fluxes of row g taken out: bit 0 north faces, bit 1 west faces
        if ((flow & 13u) || g == orow) {
            T Pc = P_land, E = T(0.000);
            if (!(on & kOnEven)) {
                keep_branch();
                const bool wet = h2 > ewl;
                Pc = wet ? P_lake : P_land;
                E = wet ? ev1t : T(0.000);
            }
            T rr = rr1t;
            if (kStorm && (on & kOnStorm)) {
                const T gy = gy_s[0][g - (r0 - 5)];
                if constexpr (kF32) rr = pk1 * gy;
                else rr = (on & kOnStorm1) ? (T)(s.st_peak * (gx1 * gy)) : T(0);
            }
            T ql = 0;
            for (int i = 0; i < nst; ++i)
                if (s.src_r[i] == g && s.src_c[i] == j) ql = (T)src_rate[2 * i];
            const T vnnPe = from_east(vnnP);
            T du = umn - umnP, dv = vnnPe - vnnP;
            if (g == orow) {
                const T h2t = (T)h2;
                qo_eff = (h2 > thh) ? T(0.5440) * h2t * M::sqrt_(gg * h2t) : T(0);
                const T du1 = qo_eff - umnP, du2 = umn - (-qo_eff);
                const T dv3 = vnnPe - (-qo_eff), dv4 = qo_eff - vnnP;
                if (out_edge <= 2) du = lanes(out_lane) ? (out_edge == 1 ? du1 : du2) : du;
                else dv = lanes(out_lane) ? (out_edge == 3 ? dv3 : dv4) : dv;
            }
            div0 = M::divc_(du, dx, rdx) + M::divc_(dv, dx, rdx);
            const T rhs = div0 - ql - rr * Pc + E;
            const TH hr = h2 - dt2h * (TH)rhs;
            D0 = vote(MH::max_(hr, TH(0.00)) < thh) & A2;
            // ---- treat_error on the faces of row g (695-725) ----
            if (D0 | D1) {
                const u64 zx = (D1 & vote(umnP > 0)) | (D0 & vote(umnP < 0));
                const u64 zy = ((D0 << 1) & vote(vnnP > 0)) | (D0 & vote(vnnP < 0));
                if (zx | zy) {
                    umpg = lanes(zx) ? T(0) : umnP;
                    vnpg = lanes(zy) ? T(0) : vnnP;
                    cut = any_lane(zx) | any_lane(zy) << 1;
                }
                if (g == orow) qo_eff = lanes(D0) ? T(0) : qo_eff;
            }
        }

        // ---- second continuity of row q = k-3 at time t + dt; store ----
        const int q = k - 3;
        TH h2v = 0;
        T src = 0;
        if (k >= r0 + 3) {
            if ((on & kOnCalm) && !(flow & 52u) && q != orow && !vote(!(h3 >= TH(0)))) {
                h2v = lanes(A3) ? h3 : TH(0);
            } else {
                T Pc = P_land, E = T(0.000);
                if (!(on & kOnEven)) {
                    keep_branch();
                    const bool wet = h3 > ewl;
                    Pc = wet ? P_lake : P_land;
                    E = wet ? ev2t : T(0.000);
                }
                T rr = rr2t;
                if (kStorm && (on & kOnStorm)) {
                    const T gy = gy_s[1][q - (r0 - 6)];
                    if constexpr (kF32) rr = pk2 * gy;
                    else rr = (on & kOnStorm2) ? (T)(s.st_peak * (gx2 * gy)) : T(0);
                }
                T ql = 0;
                for (int i = 0; i < nst; ++i)
                    if (s.src_r[i] == q && s.src_c[i] == j)
                        ql = (T)(adapt ? source_rate(s, i, st.tm) : src_rate[2 * i + 1]);
                // FP64: the divergence is the first continuity's where treat_error
                // left the row's fluxes as they were (two divisions less; in FP32
                // forming it anew costs less than the test)
                T div = div1;
                if (kF32 || (cut1 | (cut & 1u)) || q == orow) {
                    const T vnpPe = from_east(vnpP);
                    T du = umpg - umpP, dv = vnpPe - vnpP;
                    if (q == orow) {
                        const T du1 = qo_eff - umpP, du2 = umpg - (-qo_eff);
                        const T dv3 = vnpPe - (-qo_eff), dv4 = qo_eff - vnpP;
                        if (out_edge <= 2) du = lanes(out_lane) ? (out_edge == 1 ? du1 : du2) : du;
                        else dv = lanes(out_lane) ? (out_edge == 3 ? dv3 : dv4) : dv;
                    }
                    div = M::divc_(du, dx, rdx) + M::divc_(dv, dx, rdx);
                }
                const T rhs = div - ql - rr * Pc + E;
                if constexpr (kH32) {
                    // FP32 form: the depth update h3 - dt2 rhs is rounded
                    // stochastically.  TwoSum gives the exact rounding error er of
                    // sm = fl(h3 + tt); the result moves to the FP32 neighbour of sm
                    // on er's side with probability |er| / spacing, so rounding
                    // errors average out instead of adding up coherently (every
                    // cell of a uniformly wetted slope rounds the same small rain
                    // increment the same way).  The random number is a fixed hash
                    // of (cell, iteration): results are reproducible and do not
                    // depend on the tiling or on other scenarios.
                    const T tt = -dt2 * rhs;
                    const T sm = h3 + tt;
                    const T bp = sm - h3;
                    const T er = (h3 - (sm - bp)) + (tt - bp);
                    h2v = sm;
                    if (sm > T(0) && er != T(0)) {
                        const uint32_t bits = __float_as_uint(sm);
                        const T nb = __uint_as_float(er > T(0) ? bits + 1u : bits - 1u);
                        const T pr = er * __builtin_amdgcn_rcpf(nb - sm);
                        if (cell_uniform((uint32_t)(q * C + j), (uint32_t)it.step_index) < pr) h2v = nb;
                    }
                    // the exact update sm + er is negative iff sm < 0, or sm = 0 and
                    // er < 0 (|er| is at most half an ulp of sm); its FP64 value
                    // (exact: 48 bits suffice) is needed only then
                    const u64 neg = vote(sm <= T(0)) & (vote(sm < T(0)) | vote(er < T(0)));
                    if (neg) {
                        if (lanes(neg & A3)) clip_s[lane] += -((double)sm + (double)er);
                        h2v = lanes(neg) ? TH(0) : h2v;
                    }
                } else {
                    const TH hr = h3 - dt2h * (TH)rhs;
                    h2v = MH::max_(hr, TH(0.00));
                    const u64 neg = vote(hr < 0) & A3;
                    if (neg) {
                        if (lanes(neg)) clip_s[lane] += -(double)hr;
                    }
                }
                h2v = lanes(A3) ? h2v : TH(0.00);
                if constexpr (kF32) src = ql + rr * Pc - E;  // x dt2 below
                else src = st.dt2 * ((double)ql + (double)rr * (double)Pc - (double)E);
                src = lanes(A3) ? src : T(0);
            }
        }
        acc_vol += (double)h2v;
        acc_src += (double)src;
        // unconditional, for the count of accesses in flight; before the first
        // row every lane's offset is kOutside
        if (k == r0 + 3) {
            keep_branch();
            row_out = (unsigned)r0 * (unsigned)P;
            outT = colout ? (unsigned)j * (unsigned)sizeof(T) : kOutside;
            outH = colout ? (unsigned)j * (unsigned)sizeof(TH) : kOutside;
        }
        h_out.store(outH, row_out, h2v);
        um_out.store(outT, row_out, umpP);
        vn_out.store(outT, row_out, vnpP);
        row_out += k >= r0 + 3 ? (unsigned)P : 0u;

        // ---- rotate the row window ----
        push(o);
        umnP = umn; vnnP = vnn;
        umpP = umpg; vnpP = vnpg;
        D1 = D0;
        div1 = div0;
        cut1 = cut;
    }
    // the outlet's discharge, where its cell is among this tile's outputs
    double acc_q = 0;
    if (orow >= r0 && orow < r1 && lanes(out_lane & out_cols)) acc_q = (double)qo_eff * s.dy;

    // ---- per-tile partial sums (fixed-order wave reductions) ----
    double acc_clip = clip_s[lane];
    if (!lanes(out_cols)) acc_vol = acc_src = acc_clip = 0;
    if constexpr (kF32) acc_src *= st.dt2;
    acc_vol = wave_sum(acc_vol);
    acc_src = wave_sum(acc_src);
    acc_clip = wave_sum(acc_clip);
    acc_q = wave_sum(acc_q);
    double cfl = INFINITY;
    if (adapt) {
        const double m = wave_max((double)smax);
        cfl = m > 0.0 ? s.dx / m : INFINITY;
    }
    if (lane == 0) {
        Partial p;
        p.vol = acc_vol; p.src = acc_src; p.clip = acc_clip; p.qout = acc_q;
        it.part_out[tile] = p;
        if (adapt && cfl < INFINITY)
            clock_note_cfl(s.clk[it.slot_b], tile, cfl);
    }
}

// The forcing of every descriptor's current iteration, one wave a descriptor; a
// slot without a member is all zeros.  In each form's own unit: the units fuse
// multiply-adds under different rules, and a rate has to round the same here and
// where fused_step evaluates it for the next iteration.
template <typename T, typename TH>
__global__ void __launch_bounds__(64) forcing_kernel(const Scenario *scen)
{
    const StepCommon &s = scen[blockIdx.x].s;
    if (s.clk) note_forcing(s, s.slot_a, s.clk[s.slot_a].t, threadIdx.x);
}

template <typename T, typename TH>
static hipError_t launch_forcing_impl(hipStream_t stream, const Scenario *scen, int n)
{
    hipLaunchKernelGGL((forcing_kernel<T, TH>), dim3(n), dim3(64), 0, stream, scen);
    return hipGetLastError();
}

// initial CFL minimum of the state (adaptive mode)
template <typename T, typename TH>
__global__ void __launch_bounds__(256) init_cfl(const TH *h, const T *um, const T *vn,
                                                const double *z, int R, int C, int P, double dx,
                                                double dy, double g, double th, Clock *clk)
{
    using M = num<T>;
    const long n = (long)R * C;
    double cfl = INFINITY;
    for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (long)gridDim.x * blockDim.x) {
        const int r = (int)(idx / C), j = (int)(idx % C);
        const long o = (long)r * P + j;
        const bool ac = (z[o] == z[o]);
        if (r >= 1) {
            const bool an = (z[o - P] == z[o - P]);
            const TH hm = TH(0.50) * (h[o] + h[o - P]);
            if (ac && an && hm > (TH)th) {
                const T uu1 = (hm >= (TH)th) ? M::div_(um[o], (T)hm) : T(0.00);
                const double w = dx / ((double)M::abs_(uu1) + sqrt(g * (double)hm));
                cfl = (w < cfl) ? w : cfl;
            }
        }
        if (j >= 1) {
            const bool aw = (z[o - 1] == z[o - 1]);
            const TH hn = TH(0.50) * (h[o] + h[o - 1]);
            if (ac && aw && hn > (TH)th) {
                const T vv1 = (hn >= (TH)th) ? M::div_(vn[o], (T)hn) : T(0.0);
                const double w = dy / ((double)M::abs_(vv1) + sqrt(g * (double)hn));
                cfl = (w < cfl) ? w : cfl;
            }
        }
    }
    cfl = wave_min(cfl);
    if ((threadIdx.x & 63) == 0 && cfl < INFINITY)
        clock_note_cfl(clk[0], blockIdx.x, cfl);
}

// one derived field of the current state (hm_hn, uu1_vv1, uu_vv, uua_vva) over
// the cells first .. first + count - 1 of the row-major rows x cols order;
// out[i] receives cell first + i
template <typename T, typename TH>
__global__ void __launch_bounds__(256) derive_field(const TH *h, const T *um, const T *vn,
                                                    const double *z, int R, int C, int P,
                                                    double th, int field, double *out,
                                                    long first, long count)
{
    PitchedState<T, TH> ps{h, um, vn, R, C, P, (TH)th};
    const long n = first + count;
    for (long idx = first + (long)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (long)gridDim.x * blockDim.x) {
        const int r = (int)(idx / C), j = (int)(idx % C);
        const long o = (long)r * P + j;
        double v = 0;
        switch (field) {
        case SW2D_FIELD_H: v = h[o]; break;
        case SW2D_FIELD_UM: v = um[o]; break;
        case SW2D_FIELD_VN: v = vn[o]; break;
        case SW2D_FIELD_HM: v = (r == 0) ? h[o] : TH(0.50) * (h[o] + h[o - P]); break;
        case SW2D_FIELD_HN: v = (j == 0) ? h[o] : TH(0.50) * (h[o] + h[o - 1]); break;
        case SW2D_FIELD_UU1: v = ps.uu1(r, j); break;
        case SW2D_FIELD_VV1: v = ps.vv1(r, j); break;
        case SW2D_FIELD_UU: v = (h[o] >= (TH)th) ? (ps.uu1(r + 1, j) + ps.uu1(r, j)) / T(2.00) : T(0.00); break;
        case SW2D_FIELD_VV: v = (h[o] >= (TH)th) ? (ps.vv1(r, j + 1) + ps.vv1(r, j)) / T(2.00) : T(0.00); break;
        case SW2D_FIELD_UUA: v = ps.uua(r, j); break;
        case SW2D_FIELD_VVA: v = ps.vva(r, j); break;
        case SW2D_FIELD_Z: v = z[o]; break;
        default: break;
        }
        out[idx - first] = v;
    }
}

// lds: dynamic LDS bytes reserved per block and left unused (0: none); a
// batch uses it to cap the resident waves per SIMD
template <typename T, typename TH>
static hipError_t launch_fused_impl(hipStream_t stream, const Scenario *scen, const TileRef *tiles,
                                    int nblocks, int phase, int features, size_t lds)
{
    switch (fused_variant(features)) {
    case kVariant0:
        hipLaunchKernelGGL((fused_step<T, TH, kVariant0>), dim3(nblocks), dim3(64), lds, stream, scen, tiles, nblocks, phase);
        break;
    case kVariant1:
        hipLaunchKernelGGL((fused_step<T, TH, kVariant1>), dim3(nblocks), dim3(64), lds, stream, scen, tiles, nblocks, phase);
        break;
    case kVariant2:
        hipLaunchKernelGGL((fused_step<T, TH, kVariant2>), dim3(nblocks), dim3(64), lds, stream, scen, tiles, nblocks, phase);
        break;
    case kVariant3:
        hipLaunchKernelGGL((fused_step<T, TH, kVariant3>), dim3(nblocks), dim3(64), lds, stream, scen, tiles, nblocks, phase);
        break;
    default:
        hipLaunchKernelGGL((fused_step<T, TH, kFeatAll>), dim3(nblocks), dim3(64), lds, stream, scen, tiles, nblocks, phase);
        break;
    }
    return hipGetLastError();
}

// the instantiation that runs `features`
template <typename T, typename TH>
static const void *fused_fn(int features)
{
    switch (fused_variant(features)) {
    case kVariant0: return (const void *)fused_step<T, TH, kVariant0>;
    case kVariant1: return (const void *)fused_step<T, TH, kVariant1>;
    case kVariant2: return (const void *)fused_step<T, TH, kVariant2>;
    case kVariant3: return (const void *)fused_step<T, TH, kVariant3>;
    default: return (const void *)fused_step<T, TH, kFeatAll>;
    }
}

// its resident one-wave blocks per CU
template <typename T, typename TH>
static int fused_waves_per_cu_impl(int features)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fused_fn<T, TH>(features), 64, 0) != hipSuccess) return 0;
    return nb;
}

// its blocks' own LDS (the tables, the clipped volume, the storm's rows)
template <typename T, typename TH>
static size_t fused_lds_impl(int features)
{
    hipFuncAttributes a;
    if (hipFuncGetAttributes(&a, fused_fn<T, TH>(features)) != hipSuccess) return 0;
    return a.sharedSizeBytes;
}

template <typename T, typename TH>
static hipError_t launch_init_impl(sw2d_handle *h)
{
    if (!h->prm.adaptive) return hipSuccess;
    const long n = (long)h->R * h->C;
    int blocks = (int)((n + 255) / 256);
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL((init_cfl<T, TH>), dim3(blocks), dim3(256), 0, h->stream,
                       (const TH *)h->h[h->cur], (const T *)h->um[h->cur], (const T *)h->vn[h->cur],
                       (const double *)h->z, h->R, h->C, h->P, h->grid.cellsize, h->grid.cellsize,
                       h->prm.g, h->prm.th, h->clk);
    return hipGetLastError();
}

template <typename T, typename TH>
static hipError_t launch_derive_impl(sw2d_handle *h, int field, double *out_dev, long first,
                                     long count)
{
    int blocks = (int)((count + 255) / 256);
    if (blocks > 8192) blocks = 8192;
    if (blocks < 1) return hipSuccess;
    hipLaunchKernelGGL((derive_field<T, TH>), dim3(blocks), dim3(256), 0, h->stream,
                       (const TH *)h->h[h->cur], (const T *)h->um[h->cur], (const T *)h->vn[h->cur],
                       (const double *)h->z, h->R, h->C, h->P, h->prm.th, field, out_dev, first,
                       count);
    return hipGetLastError();
}

}  // namespace sw2d
