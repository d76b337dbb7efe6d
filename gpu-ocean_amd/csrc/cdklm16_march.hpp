// cdklm16_march.hpp -- one CDKLM16 Runge-Kutta substep, column-marching form.
//
// Device code for gfx950, constant Coriolis parameter and zero grid rotation
// (north = (0, 1)), the configuration of every benchmark workload.  The
// arithmetic is the one of cdklm16_tile.hpp (the reference's operand order
// and rounding points of gpu_ocean/SWESimulators/gpu_kernels/
// CDKLM16_kernel.cu:80-1006, correctly rounded division and square root), so
// the two kernels give the same bits; what differs is how work is laid out:
//
//   * one wavefront owns a strip of 64 padded columns (lane = column) and
//     walks up bh output rows; lanes 2..61 write output, lanes 0, 1, 62, 63
//     are the strip's x halo;
//   * every per-row quantity is formed once per lane and kept in registers
//     while it is needed: the converted (eta, u, v) of the last three rows,
//     the y slopes of the last two, the corner depths of the last four, and
//     the flux through the lane's north face, which is the next row's south
//     face -- so the y direction needs no data exchange at all;
//   * the x neighbours (left and right lane) are whole-wave shifts by one
//     lane (DPP), vector instructions without LDS or barriers;
//   * boundary handling is per lane (the column's wall mirror / periodic
//     wrap, fixed for the whole strip) or per row (uniform over the wave), so
//     interior and boundary strips run the same code with no per-cell index
//     arithmetic; loads address one uniform row pointer plus the lane's
//     32-bit column offset;
//   * no LDS, no __syncthreads: each wave is independent and the occupancy
//     is set by vector registers alone.
//
// What bounds it: vector issue.  A wave issues one instruction (vector,
// scalar or memory) in about 2.4 ns; a SIMD with three or more waves issues a
// float add, multiply or fma on vector registers every 1.05 ns and a compare,
// min / max, select, or any instruction with a scalar-register source every
// 1.8 ns, a reciprocal or square root every 3.5 ns.  So small domains (about
// one wave per SIMD) take 1.13 us per row whatever else happens, and large
// ones about 0.5 us per row and SIMD; fewer instructions of either kind help
// both.  Hence the wave-uniform fast paths (one compare into a scalar mask
// decides for the row), constants in vector registers, and rare rows, strips
// and depths kept in branches of their own.  2048 x 2048, SSP-RK2, 15 rows per
// strip: 50.9 us per substep before these, 44.7 us after (491 to 410 vector
// instructions per cell).
//
// Work per output cell: the tile kernel converts (BH+4)(BW+4)-4*4 cells for
// BW*BH outputs and forms every x and y quantity on its halo; here every
// quantity is formed 64/60 times per output, plus a prologue of four
// conversions, two y slopes and a face per strip of bh rows.  The host picks
// bh so that the strips fill whole rounds of resident waves (march_rows).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cdklm16_tile.hpp"

namespace gocean {
namespace march {

constexpr int kLanes = 64;
constexpr int kOut = 60;          // output columns per strip (lanes 2..61)

// index of the wavefront within its workgroup, as a scalar: everything
// derived from it (strip, rows, row addresses) stays in scalar registers
__device__ __forceinline__ int wave_in_group() {
    return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// value of `v` in the lane below / above (the neighbour column), as a whole
// wave shift by one (DPP wave_shr:1 / wave_shl:1): a vector instruction,
// often folded into the one that uses the value, where ds_bpermute is a
// round trip through the LDS pipe.  The lane past the end reads zero; what
// lanes 0 and 63 form from it is never used.
__device__ __forceinline__ float from_left(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xF, 0xF, true));
}
__device__ __forceinline__ float from_right(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xF, 0xF, true));
}

// Each plane is addressed as a wave-uniform row address (scalar registers:
// the plane's base plus the row's byte offset) plus the lane's column byte
// offset (a vector register fixed for the strip), so a row's loads and
// stores take no vector address arithmetic.
using rsrc_t = const float*;

__device__ __forceinline__ rsrc_t plane(const float* p) { return p; }
// The row address, held in scalar registers and opaque to the optimizer:
// without this, loop-invariant code motion regroups (plane + row) + lane
// into (plane + lane) + row, which costs a 64-bit vector add per access
// and two vector registers per plane.  The empty asm emits no instruction.
using gchar = __attribute__((address_space(1))) char;     // global memory
__device__ __forceinline__ gchar* srow(rsrc_t r, uint32_t row_off) {
    gchar* row = (gchar*)(const_cast<char*>(reinterpret_cast<const char*>(r))) + row_off;
    asm("" : "+s"(row));
    return row;
}
// a wave-uniform flag as an opaque 32-bit scalar: held across the row loop
// in one scalar register and tested with a scalar compare, where a bool
// would be kept as a 64-bit lane mask (and spilled under register pressure)
__device__ __forceinline__ int sflag(bool b) {
    int v = __builtin_amdgcn_readfirstlane(b ? 1 : 0);   // float compares give a vector result
    asm("" : "+s"(v));
    return v;
}

// a launch constant in a vector register, opaque to the optimizer.  On this
// chip a float add, multiply or fma issues in half the cycles when none of
// its operands is a scalar register (measured, many waves per SIMD: 1.05 ns
// against 1.78 ns per wave instruction), and the row loop has about 55 that
// take a constant; compares, min / max and med3 take the longer time either
// way, so their thresholds stay scalar.
__device__ __forceinline__ void vconst(float& v) { asm("" : "+v"(v)); }

// the lane's 32-bit offset, zero-extended at each access (scalar base plus
// 32-bit vector offset is the load's addressing form)
__device__ __forceinline__ uint32_t voff(uint32_t lane_off) {
    asm("" : "+v"(lane_off));
    return lane_off;
}
__device__ __forceinline__ float ld(rsrc_t r, uint32_t lane_off, uint32_t row_off) {
    return *(const __attribute__((address_space(1))) float*)(srow(r, row_off) + voff(lane_off));
}
__device__ __forceinline__ void st(rsrc_t r, uint32_t lane_off, uint32_t row_off, float v) {
    *(__attribute__((address_space(1))) float*)(srow(r, row_off) + voff(lane_off)) = v;
}

// corner depth with land flagged (CDKLM16_kernel.cu:509-525)
__device__ __forceinline__ float flag_land(float h, const Consts& K) {
    return (fabsf(h - K.land) < kDryEps) ? kDryFlag : h;
}

// no active lane has c: one compare into a scalar mask (__all would first
// turn the condition into a vector of 0 / 1, two more vector instructions)
__device__ __forceinline__ bool none(bool c) { return __builtin_amdgcn_ballot_w64(c) == 0ull; }

// every lane of `lanes` has a and b above c, and neither is NaN: two compares
// and a scalar or (a compare of fminf(a, b), as many vector instructions, would
// drop a NaN -- the face depth of a dry cell with an infinite corner is one)
__device__ __forceinline__ bool both_above(float a, float b, float c, unsigned long long lanes) {
    return ((__builtin_amdgcn_ballot_w64(!(a > c)) | __builtin_amdgcn_ballot_w64(!(b > c))) & lanes) == 0ull;
}

__device__ __forceinline__ bool is_inf(float v) { return fabsf(v) == INFINITY; }

// marks code that few rows or strips run: the empty volatile asm keeps the
// compiler from executing it unconditionally behind selects
__device__ __forceinline__ void rare() { asm volatile(""); }

// lanes whose slope centres (1..62) and whose y faces (2..61) are used; what
// the others compute from wrapped neighbours never decides a path
constexpr unsigned long long kSlopeLanes = 0x7FFFFFFFFFFFFFFEull;
constexpr unsigned long long kOutLanes = 0x3FFFFFFFFFFFFFFCull;

// one row of corner depths (hc, hn) = Hi[R][C], Hi[R][C+1]: land flagged;
// true when every lane's are plain (SubstepDerived::plain_hi)
__device__ __forceinline__ bool corner_row(float& hc, float& hn, const Consts& K) {
    if ((__builtin_amdgcn_ballot_w64(!(fmaxf(hc, hn) < K.plain_hi)) |
         __builtin_amdgcn_ballot_w64(!(fminf(hc, hn) > kDryFlag))) == 0ull)
        return true;
    rare();
    hc = flag_land(hc, K);
    hn = flag_land(hn, K);
    return false;
}

// converted state of one cell: (eta, u, v) with dry / land handling, the
// cell depth as the update uses it (0.25 * the corner sum), and the sum of
// its two west corners
struct Cell {
    float E, U, V, Hm4, ab;
};

// (:546-602, initBm :84-105).  a = Hi[R][C], b = Hi[R+1][C], c = Hi[R][C+1],
// d = Hi[R+1][C+1] (land flagged); plain: both corner rows are plain.
// dry: set when a lane of kSlopeLanes holds the dry flag in E.
__device__ __forceinline__ Cell convert(float eta, float hu, float hv, float a, float b, float c, float d,
                                        bool plain, const Consts& K, int& dry) {
    Cell o;
    o.ab = a + b;
    const float sum = (o.ab + c) + d;
    o.Hm4 = sum * 0.25f;
    float Hm = o.Hm4;
    const float h = eta + Hm;
    // every lane wet and deep: the plain branch alone
    if (plain && none(h < K.desing)) {
        o.E = eta;
        const float rh = rcp_refined(h);
        o.U = div_r(hu, h, rh);
        o.V = div_r(hv, h, rh);
    } else {
        rare();
        const bool any_dry = (a == kDryFlag) | (b == kDryFlag) | (c == kDryFlag) | (d == kDryFlag);
        if (any_dry) {
            const float wet = 4.0f - (float)(a == kDryFlag) - (float)(b == kDryFlag)
                            - (float)(c == kDryFlag) - (float)(d == kDryFlag);
            Hm = (wet == 0.0f) ? K.land : sum / wet;
        }
        const float hh = eta + Hm;
        if (fabsf(Hm - K.land) <= kDryEps) {
            o.E = kDryFlag; o.U = 0.0f; o.V = 0.0f;
        } else if (hh < K.desing) {
            if (hh <= K.cutoff) {
                o.E = -Hm + K.cutoff; o.U = 0.0f; o.V = 0.0f;
            } else {
                o.E = eta;
                o.U = desingularize(hh, hu, K.desing);
                o.V = desingularize(hh, hv, K.desing);
            }
        } else {
            o.E = eta;
            const float rh = rcp_refined(hh);
            o.U = div_r(hu, hh, rh);
            o.V = div_r(hv, hh, rh);
        }
    }
    dry = (__builtin_amdgcn_ballot_w64(o.E == kDryFlag) & kSlopeLanes) != 0ull;
    return o;
}

// The backward candidates of a cell's three minmod slopes equal, bit for
// bit, the forward candidates of its low-side neighbour: (c - l) * theta of
// the cell is (r - c) * theta of the neighbour, and the geostrophic candidate
// theta g ((e_c - e_l) -+ d/(2g) (f_c + f_l)) is the neighbour's forward one
// up to the order of the commutative sum f_c + f_l.  So each slope centre
// takes them from its neighbour (the previous row in y, the left lane in x)
// and hands its own forward ones on.
struct Carry {
    float a;     // (a_c - a_l) * theta
    float b;     // (b_c - b_l) * theta
    float K;     // geostrophic backward candidate
    float fb;    // f * b_l (with b_l's wall flip)
};

// forward candidates of one cell (x: :607-666 with adjustSlopes_x :148-191;
// y: :711-770 with adjustSlopes_y :198-241), zero-rotation form.  c, r: the
// cell and its high neighbour along the direction; `a` the velocity along
// the direction (minmod only), `b` the velocity in the geostrophic term (v
// for x, u for y); fc, fr: f * b of the two with their wall flips (the flip
// goes into the sign of f, once per strip or row: the same product).  SGN -1
// for x, +1 for y (the sign of the geostrophic term).
template <int SGN>
__device__ __forceinline__ Carry slope_fwd(float ec, float er, float ac, float ar, float bc, float br,
                                           float fc, float fr, float vd, const Consts& K) {
    Carry o;
    o.a = (ar - ac) * K.theta;
    o.b = (br - bc) * K.theta;
    o.fb = fc;
    if constexpr (SGN < 0) o.K = K.theta_g * ((er - ec) - vd * (fc + fr));
    else o.K = K.theta_g * ((er - ec) + vd * (fc + fr));
    return o;
}

// Slope centre of one cell: minmod slopes Sa, Sb, T = (K + d f v)/2g (x) or
// (L - d f u)/2g (y), and the depths of the cell's two faces as the face
// fluxes form them, dlo = (e + H_lo) - T and dhi = (e + H_hi) + T.  Hlo2,
// Hhi2: corner sums of the faces, twice their averaged depths (0.5 * Hlo2 is
// exact, so one fma rounds as the sum e + H does); dfb = d f b with the
// adjustment's own flip; `fix`: some lane's wall flip differs from the
// adjustment's (a scalar), and in the lane itself flc != fa, with db = d f b
// under the slope's own flip.  `in`: the backward candidates (from the low
// neighbour); `out`: this cell's forward ones.  ok: every lane of `lanes`
// has both face depths above face_lo (so no adjustment fired and both
// faces are wet on this side).
// REC: also the slope centre's branch record (tape code byte): the minmod
// selections of the u and v slopes and of K / L, and which positivity
// adjustment fired (x: a = u; y: a = v).
template <int SGN, bool FAST, bool REC = false>
__device__ __forceinline__ void slope_rest(float el, float ec, float er, float al, float ar, float bl, float br,
                                           float Hlo2, float Hhi2, bool fix, bool lane_fix, float dfb, float db,
                                           float vd, const Consts& K, float fr,
                                           unsigned long long lanes, const Carry& in, const Carry& out,
                                           float& Sa, float& Sb, float& T, float& dlo, float& dhi, int& ok,
                                           uint32_t* code8 = nullptr) {
    const float ca = (ar - al) * 0.5f, cb = (br - bl) * 0.5f;
    Sa = minmod3(in.a, ca, out.a);
    Sb = minmod3(in.b, cb, out.b);
    float ce;
    if constexpr (SGN < 0) ce = K.half_g * ((er - el) - vd * (fmaf(2.0f, out.fb, fr) + in.fb));
    else ce = K.half_g * ((er - el) + vd * (fmaf(2.0f, out.fb, fr) + in.fb));
    float Kv = minmod3(in.K, ce, out.K);
    const float elo = fmaf(0.5f, Hlo2, ec), ehi = fmaf(0.5f, Hhi2, ec);
    T = (SGN < 0) ? div_k<FAST>(Kv + dfb, K.two_g, K.r_two_g, K.l_two_g)
                  : div_k<FAST>(Kv - dfb, K.two_g, K.r_two_g, K.l_two_g);
    dlo = elo - T;
    dhi = ehi + T;
    if constexpr (REC) {
        if (FAST && is_inf(T)) T = dlo = dhi = NAN;
        const uint32_t sa = minmod_sel(in.a, ca, out.a);
        const uint32_t sb = minmod_sel(in.b, cb, out.b);
        const uint32_t sk = minmod_sel(in.K, ce, out.K);
        const uint32_t ad = !(dhi > 0.0f) ? 2u : (!(dlo > 0.0f) ? 1u : 0u);
        *code8 = (SGN < 0 ? (sa | (sb << 2)) : (sb | (sa << 2))) | (sk << 4) | (ad << 6);
    }
    ok = both_above(dlo, dhi, K.face_lo, lanes);
    if (!ok || fix) {
        rare();
        // past 1e37 the numerators overflow; an infinite T (one of the depths
        // is then -inf or NaN, so the row comes here) is NaN as in div_r
        if (FAST && is_inf(T)) T = dlo = dhi = NAN;
        bool adj = false;
        const bool alo = !(dlo > 0.0f), ahi = !(dhi > 0.0f);
        if constexpr (SGN < 0) {
            if (alo) { Kv = (-dfb) + K.two_g * elo; adj = true; }
            if (ahi) { Kv = (-dfb) - K.two_g * ehi; adj = true; }
        } else {
            if (alo) { Kv = dfb + K.two_g * elo; adj = true; }
            if (ahi) { Kv = dfb - K.two_g * ehi; adj = true; }
        }
        if (adj || lane_fix) {
            T = (SGN < 0) ? div_k<FAST>(Kv + db, K.two_g, K.r_two_g, K.l_two_g)
                          : div_k<FAST>(Kv - db, K.two_g, K.r_two_g, K.l_two_g);
            if (FAST && is_inf(T)) T = NAN;
            dlo = elo - T;
            dhi = ehi + T;
        }
        ok = both_above(dlo, dhi, K.face_lo, lanes);
    }
}

// one face between cell m (low side) and p (high side) (:246-370):
// reconstructed states and central-upwind flux.  Sa*, Sb*: the minmod slopes
// (half of them is exact, so one fma rounds as a +- 0.5 S does); dm / dp: the
// face depths (e + H_face) + T of m and (e + H_face) - T of p before the
// clamp at zero, as the slope centres formed them.  For x faces (a, b) =
// (u, v) and the result is (F.x, F.y, F.z); for y faces (a, b) = (v, u) and
// the flux comes back as (G.x, G.z, G.y) -- the caller swaps, as the
// reference's computeGFaceFlux does.  wet (wave-uniform): no used lane's face
// touches a dry-flagged cell and all face depths are above face_lo; then the
// same operations run without the clamps and the selects of the dry and
// zero-flux cases (and, with FAST, the wave speeds take the Newton square
// root: both depths are above the cutoff there).
// REC: also the face's branch record (which states give a+ and a-, and
// the zero-flux bit), as cu_flux<true>.
template <bool FAST, bool REC = false>
__device__ __forceinline__ void face(bool wet, float em, float am, float bm, float Sam, float Sbm, float dm,
                                     float ep, float ap, float bp, float Sap, float Sbp, float dp,
                                     const Consts& K, float& F0, float& F1, float& F2, uint32_t* code = nullptr) {
    const float up = fmaf(-0.5f, Sap, ap), vp = fmaf(-0.5f, Sbp, bp);
    const float um = fmaf(0.5f, Sam, am), vm = fmaf(0.5f, Sbm, bm);
    if (wet) {
        const float hp = dp, hm = dm;
        const float qp = hp * up;
        const float Fpx = qp, Fpy = qp * up + (K.half_g * hp) * hp, Fpz = qp * vp;
        const float c_p = sqrt_k<FAST>(K.g * hp);
        const float qm = hm * um;
        const float Fmx = qm, Fmy = qm * um + (K.half_g * hm) * hm, Fmz = qm * vm;
        const float c_m = sqrt_k<FAST>(K.g * hm);
        const float amin = fminf(fminf(um - c_m, up - c_p), 0.0f);
        const float amax = fmaxf(fmaxf(um + c_m, up + c_p), 0.0f);
        const float den = amax - amin;
        if constexpr (REC) {
            const float b1 = um + c_m, b2 = up + c_p, a1 = um - c_m, a2 = up - c_p;
            const uint32_t cp = (fmaxf(b1, b2) > 0.0f) ? ((b1 >= b2) ? 1u : 2u) : 0u;
            const uint32_t cm = (fminf(a1, a2) < 0.0f) ? ((a1 <= a2) ? 1u : 2u) : 0u;
            *code = cp | (cm << 2);
        }
        const float apam = amax * amin;
        const float rden = rcp_refined(den);
        F0 = div_r((amax * Fmx - amin * Fpx) + apam * (hp - hm), den, rden);
        F1 = div_r((amax * Fmy - amin * Fpy) + apam * (Fpx - Fmx), den, rden);
        F2 = (um + up > 0.0f) ? Fmz : Fpz;
        return;
    }
    rare();
    F0 = 0.0f; F1 = 0.0f; F2 = 0.0f;
    if constexpr (REC) *code = 0u;
    if (!(ep == kDryFlag || em == kDryFlag))
        cu_flux<REC>(fmaxf(0.0f, dm), um, vm, fmaxf(0.0f, dp), up, vp, K, F0, F1, F2, code);
}

// One strip: padded columns sx*60 .. sx*60+63 (lanes), output rows
// 2 + sy*bh .. min(2 + (sy+1)*bh, ny+2) - 1.  WGRID: the wind stress comes
// from A.wind_grid (else the uniform A.wind_x, A.wind_y); a separate
// instantiation, because the per-lane interpolation state and lookups would
// otherwise hold registers in every launch.  STAGE: the first or second stage
// of an order 1 / 2 step without friction, or any (decided at run time); the
// two common ones carry no scalar registers or branches for the others.
// REC: also write the branch
// record (A.tape_*) of the reverse pass, the same words the tile kernel's
// recording variant writes.
enum { kStageFirst = 0, kStageSecond = 1, kStageAny = 2 };

template <bool FAST, bool WGRID, int STAGE, bool REC = false>
__device__ __forceinline__ void march_strip(const SubstepArgs& A, int sx, int sy, int bh) {
    const int lane = threadIdx.x & (kLanes - 1);
    const int nx = A.nx, ny = A.ny;
    const uint32_t rowb = (uint32_t)A.pitch * 4u, hrowb = (uint32_t)A.hi_pitch * 4u;   // row bytes
    Consts K = make_consts(A);
    float fcor = A.f, dt = A.dt_dev ? *A.dt_dev : A.dt;
    vconst(K.theta); vconst(K.theta_g); vconst(K.half_g); vconst(K.g); vconst(K.vdx); vconst(K.udy);
    vconst(K.r_two_g); vconst(K.l_two_g); vconst(K.r_dx); vconst(K.l_dx); vconst(K.r_dy); vconst(K.l_dy);
    vconst(K.dyf); vconst(fcor); vconst(dt);
    const int C = sx * kOut + lane;                  // padded column of the lane
    const int Cl = min(C, nx + 3);                   // load column (clamped)
    const int j0 = 2 + sy * bh;
    const int j1 = min(j0 + bh, ny + 2);
    const int wN = sflag(A.bc_n() == kWall), wS = sflag(A.bc_s() == kWall);
    const bool wE = A.bc_e() == kWall, wW = A.bc_w() == kWall;
    const int pNS = sflag(A.bc_n() == kPeriodic), pEW = sflag(A.bc_e() == kPeriodic);

    // the lane's source column (wall mirror with u negated, or periodic wrap)
    int sc = Cl;
    bool neg_u = false;
    if (Cl < 2) {
        if (wW) { sc = 3 - Cl; neg_u = true; } else if (pEW) { sc = Cl + nx; }
    } else if (Cl > nx + 1) {
        if (wE) { sc = 2 * nx + 3 - Cl; neg_u = true; } else if (pEW) { sc = Cl - nx; }
    }
    auto col_flip = [&](int c) { return (wW && c < 2) || (wE && c > nx + 1); };
    // the wall flips of the geostrophic velocity go into the sign of f, once
    // per strip (x) or row (y): f * (-v) and (-f) * v are the same float
    const bool xfc = col_flip(C);
    const bool xfa = wW && C < 2;
    const float fx = xfc ? -fcor : fcor;               // slope and face term
    const float dfx = xfa ? -K.dxf : K.dxf;   // positivity adjustment
    const int xfix = sflag((__builtin_amdgcn_ballot_w64(xfc != xfa) & kSlopeLanes) != 0ull);
    auto row_flip = [&](int r) { return (wS && r < 2) || (wN && r > ny + 1); };
    auto times_f = [&](float u, int r) {
        float v = fcor * u;
        if (row_flip(r)) { rare(); v = -v; }
        return v;
    };
    const int any_neg = sflag(!none(neg_u));
    const int hc = min(C, nx + 4), hn = min(C + 1, nx + 4);   // corner-depth columns
    // byte offsets of the lane's columns within a row
    const uint32_t osc = (uint32_t)sc * 4u, ohc = (uint32_t)hc * 4u, ohn = (uint32_t)hn * 4u;
    const uint32_t ocl = (uint32_t)Cl * 4u;
    const rsrc_t r_ein = plane(A.eta_in), r_uin = plane(A.hu_in), r_vin = plane(A.hv_in);
    const rsrc_t r_hi = plane(A.Hi);
    // branch record: each cell's words are written by one strip -- interior
    // columns by lanes 2..61, the ghost columns by the first and last strip
    // (ghost corners are never written, as in the tile kernel)
    const bool col_in = C >= 2 && C <= nx + 1;
    const bool rec_lane = REC && (col_in ? (lane >= 2 && lane <= 61)
                                         : (C <= 1 ? sx == 0 : (C <= nx + 3 && sx == A.tiles_x - 1)));
    auto rec_store = [&](int R, float u, float v) {
        const uint32_t ro = (uint32_t)R * rowb;
        st(plane(A.tape_u), ocl, ro, u);
        st(plane(A.tape_v), ocl, ro, v);
    };
    auto rec_code = [&](int R, uint32_t code) {
        st(plane(reinterpret_cast<const float*>(A.tape_code)), ocl, (uint32_t)R * rowb, __uint_as_float(code));
    };


    // state row R of the input (remapped) and the corner-depth row R
    auto load_state = [&](int R, float& e, float& u, float& v) {
        int sr = R;
        bool neg_v = false;
        if (R < 2) {
            if (wS) { sr = 3 - R; neg_v = true; } else if (pNS) { sr = R + ny; }
        } else if (R > ny + 1) {
            if (wN) { sr = 2 * ny + 3 - R; neg_v = true; } else if (pNS) { sr = R - ny; }
        }
        const uint32_t ro = (uint32_t)sr * rowb;
        e = ld(r_ein, osc, ro);
        u = ld(r_uin, osc, ro);
        v = ld(r_vin, osc, ro);
        if (any_neg) { rare(); u = neg_u ? -u : u; }
        if (neg_v) { rare(); v = -v; }
    };
    // the same for the rows of the row loop, R >= 4: only the rows past the
    // north side are remapped
    auto load_next = [&](int R, float& e, float& u, float& v) {
        int sr = R;
        if (R > ny + 1) {
            rare();
            sr = wN ? 2 * ny + 3 - R : (pNS ? R - ny : R);
        }
        const uint32_t ro = (uint32_t)sr * rowb;
        e = ld(r_ein, osc, ro);
        u = ld(r_uin, osc, ro);
        v = ld(r_vin, osc, ro);
    };
    auto load_hi = [&](int R, float& a, float& b) {
        const uint32_t ro = (uint32_t)R * hrowb;
        a = ld(r_hi, ohc, ro);
        b = ld(r_hi, ohn, ro);
    };

    // ---- prologue: conversion of rows j0-2 .. j0+1, y slopes of rows
    //      j0-1 and j0, the flux through the face (j0-1 | j0) ----
    Cell c0, c1, c2, c3;                             // rows j0-2, j0-1, j0, j0+1
    int dry1, dry2, dry3;                            // a used lane of rows j0-1 .. j0+1 is dry-flagged
    float hcE, hnE;                                  // corner row j0+2
    bool plE;
    float Hs_m1, Hs_0, Hs_1;                         // corner sums of rows j0-1, j0, j0+1 (twice the south face depths)
    {
        float hcA, hnA, hcB, hnB, hcC, hnC, hcD, hnD;
        float e0, u0, v0, e1, u1, v1, e2, u2, v2, e3, u3, v3;
        load_hi(j0 - 2, hcA, hnA);
        load_hi(j0 - 1, hcB, hnB);
        load_state(j0 - 2, e0, u0, v0);
        load_hi(j0, hcC, hnC);
        load_state(j0 - 1, e1, u1, v1);
        load_hi(j0 + 1, hcD, hnD);
        load_state(j0, e2, u2, v2);
        load_hi(j0 + 2, hcE, hnE);
        load_state(j0 + 1, e3, u3, v3);
        const bool plA = corner_row(hcA, hnA, K), plB = corner_row(hcB, hnB, K);
        int dry0;
        c0 = convert(e0, u0, v0, hcA, hcB, hnA, hnB, plA && plB, K, dry0);
        const bool plC = corner_row(hcC, hnC, K);
        c1 = convert(e1, u1, v1, hcB, hcC, hnB, hnC, plB && plC, K, dry1);
        const bool plD = corner_row(hcD, hnD, K);
        c2 = convert(e2, u2, v2, hcC, hcD, hnC, hnD, plC && plD, K, dry2);
        plE = corner_row(hcE, hnE, K);
        c3 = convert(e3, u3, v3, hcD, hcE, hnD, hnE, plD && plE, K, dry3);
        Hs_m1 = hcB + hnB;
        Hs_0 = hcC + hnC;
        Hs_1 = hcD + hnD;
    }
    // y slopes of row j0-1 (cells c0, c1, c2) and row j0 (c1, c2, c3); in y
    // (a, b) = (v, u)
    float Uy1, Vy1, S1, dhi1;
    int oky1;                                        // row j0's y face depths are all above face_lo
    Carry ycar;
    float gsx, gsy, gsz;
    uint32_t yc1 = 0u;                               // record byte of row j0's y slope centre
    {
        float Uy0, Vy0, S0, dlo0, dhi0, dlo1;
        int oky0;
        uint32_t yc0 = 0u, gc0 = 0u;
        const float f0 = times_f(c0.U, j0 - 2), f1 = times_f(c1.U, j0 - 1), f2 = times_f(c2.U, j0), f3 = times_f(c3.U, j0 + 1);
        // the backward candidates of row j0-1 are row j0-2's forward ones
        const Carry bwd = slope_fwd<+1>(c0.E, c1.E, c0.V, c1.V, c0.U, c1.U, f0, f1, K.udy, K);
        const Carry fwd = slope_fwd<+1>(c1.E, c2.E, c1.V, c2.V, c1.U, c2.U, f1, f2, K.udy, K);
        const bool fa0 = wS && j0 - 1 < 2, fl0 = row_flip(j0 - 1);
        slope_rest<+1, FAST, REC>(c0.E, c1.E, c2.E, c0.V, c2.V, c0.U, c2.U, Hs_m1, Hs_0, fl0 != fa0, fl0 != fa0,
                                  c1.U * (fa0 ? -K.dyf : K.dyf), c1.U * (fl0 ? -K.dyf : K.dyf), K.udy, K, f2,
                                  kOutLanes, bwd, fwd, Vy0, Uy0, S0, dlo0, dhi0, oky0, &yc0);
        const Carry fwd1 = slope_fwd<+1>(c2.E, c3.E, c2.V, c3.V, c2.U, c3.U, f2, f3, K.udy, K);
        // row j0 is an interior row: no flips of its own
        slope_rest<+1, FAST, REC>(c1.E, c2.E, c3.E, c1.V, c3.V, c1.U, c3.U, Hs_0, Hs_1, false, false,
                                  c2.U * K.dyf, c2.U * K.dyf, K.udy, K, f3,
                                  kOutLanes, fwd, fwd1, Vy1, Uy1, S1, dlo1, dhi1, oky1, &yc1);
        ycar = fwd1;
        // flux through (j0-1 | j0): m = row j0-1 (c1), p = row j0 (c2)
        float a, b, c;
        face<FAST, REC>(oky0 && oky1 && !dry1 && !dry2, c1.E, c1.V, c1.U, Vy0, Uy0, dhi0, c2.E, c2.V, c2.U, Vy1, Uy1,
                        dlo1, K, a, b, c, &gc0);
        gsx = a; gsy = c; gsz = b;
        // the first strip of a column records ghost rows 0 and 1 (interior
        // columns; row 1's y slope centre and its north face (1 | 2))
        if (REC && sy == 0 && rec_lane && col_in) {
            rec_store(0, c0.U, c0.V);
            rec_code(0, 0u);
            rec_store(1, c1.U, c1.V);
            st(plane(A.tape_s), ocl, rowb, S0);
            rec_code(1, (yc0 << kCodeY) | (gc0 << kCodeFy));
        }
    }
    // window: (cj, cj1) = rows j, j+1; (Uyj, Vyj, Sj, dhij, okyj) = y slopes,
    // depth term, north-face depth and wet flag of row j; ycar = forward
    // candidates of row j; (hc2, hn2, pl2) = corner row j+2; Hsj, Hnj =
    // corner sums of rows j and j+1 (twice the depths of row j's south and
    // north faces)
    Cell cj = c2, cj1 = c3;
    float Uyj = Uy1, Vyj = Vy1, Sj = S1, dhij = dhi1;
    int okyj = oky1, dryj = dry2, dryj1 = dry3;
    float hc2 = hcE, hn2 = hnE;
    int pl2 = plE;
    float Hsj = Hs_0, Hnj = Hs_1;
    const int friction = STAGE == kStageAny ? sflag(A.r > 0.0f) : 0;
    // gridded wind: the lane's column weights, fixed for the strip
    constexpr bool wgrid = WGRID;
    WindAxis wax;
    wax.i0 = wax.i1 = 0; wax.a = 0.0f;
    if (wgrid) wax = wind_axis(C, nx, A.wind_wx);
    const int rk_order = STAGE == kStageAny ? A.rk_order() : 2;
    const int rk_step = STAGE == kStageAny ? A.rk_step() : STAGE;
    const bool later = STAGE == kStageAny ? rk_step > 0 : STAGE == kStageSecond;   // reads Q^n
    const bool store_lane = lane >= 2 && lane < 2 + kOut && C <= nx + 1;
    // the strip has output columns with periodic images
    const int ghost_cols = sflag(pEW && (__builtin_amdgcn_ballot_w64(store_lane && (C <= 3 || C >= nx)) != 0ull));
    const rsrc_t r_eqn = plane(A.eta_qn), r_uqn = plane(A.hu_qn), r_vqn = plane(A.hv_qn);
    const rsrc_t r_eo = plane(A.eta_out), r_uo = plane(A.hu_out), r_vo = plane(A.hv_out);

    uint32_t ycj = yc1;                               // record byte of row j's y slope centre
    for (int j = j0; j < j1; ++j) {
        // loads for row j+2 (conversion) and Q^n of row j (second stages)
        float e2, u2, v2, hc3, hn3;
        load_next(j + 2, e2, u2, v2);
        load_hi(j + 3, hc3, hn3);
        const uint32_t rj = (uint32_t)j * rowb;
        float ea = 0.0f, ha = 0.0f, va = 0.0f;
        if (later) { ea = ld(r_eqn, ocl, rj); ha = ld(r_uqn, ocl, rj); va = ld(r_vqn, ocl, rj); }

        // the gridded wind's 16 texels of the lane's cell: in flight until
        // the sources at the end of the row
        WindCell wcell;
        if (wgrid) wcell = wind_grid_load(A.wind_grid, A.wind_wx, A.wind_wy, wax, wind_axis(j, ny, A.wind_wy));

        // ---- x slope centre of row j (neighbours by lane exchange) ----
        const float el = from_left(cj.E), er = from_right(cj.E);
        const float ul = from_left(cj.U), ur = from_right(cj.U);
        const float vl = from_left(cj.V), vr = from_right(cj.V);
        const float Hw2 = cj.ab;                         // corner sum of the west face
        const float He2 = from_right(Hw2);         // of the east face
        float Ux, Vx, T, dlox, dhix;
        int okx;
        uint32_t xc = 0u, fce = 0u, ycn = 0u, gcn = 0u;   // record bytes of row j (x, east face, north face), row j+1 (y)
        {
            const float fbc = cj.V * fx;
            const float fbr = from_right(fbc);
            const Carry fwd = slope_fwd<-1>(cj.E, er, cj.U, ur, cj.V, vr, fbc, fbr, K.vdx, K);
            Carry bwd;
            bwd.a = from_left(fwd.a);
            bwd.b = from_left(fwd.b);
            bwd.K = from_left(fwd.K);
            bwd.fb = from_left(fwd.fb);
            slope_rest<-1, FAST, REC>(el, cj.E, er, ul, ur, vl, vr, Hw2, He2, xfix, xfc != xfa, cj.V * dfx,
                                      K.dxf * (xfc ? -cj.V : cj.V), K.vdx, K, fbr, kSlopeLanes, bwd, fwd,
                                      Ux, Vx, T, dlox, dhix, okx, &xc);
        }
        // ---- east face (C | C+1) ----
        const float Uxr = from_right(Ux), Vxr = from_right(Vx), dpr = from_right(dlox);
        float fex, fey, fez;
        face<FAST, REC>(okx && !dryj, cj.E, cj.U, cj.V, Ux, Vx, dhix, er, ur, vr, Uxr, Vxr, dpr, K, fex, fey, fez,
                        &fce);

        // ---- conversion of row j+2, y slopes of row j+1, north face ----
        // the north wall's flips concern the last two rows of the domain
        const bool north = j >= ny && wN;
        if (any_neg) { rare(); u2 = neg_u ? -u2 : u2; }
        if (north) { rare(); v2 = -v2; }
        const bool pl3 = corner_row(hc3, hn3, K);
        int dryj2;
        const Cell cj2 = convert(e2, u2, v2, hc2, hc3, hn2, hn3, pl2 && pl3, K, dryj2);
        const float Hnj1 = hc2 + hn2;                    // corner sum of row j+1's north face
        float Uyn, Vyn, Sn, dlon, dhin;
        int okyn;
        {
            float fbc = fcor * cj1.U, fbr = fcor * cj2.U, db = cj1.U * K.dyf;
            const float dfb = db;
            // row j+1 is interior or the first north ghost row, whose wall
            // flip the adjustment does not take
            bool fix = false;
            if (north) {
                rare();
                fbr = -fbr;
                if (j + 1 > ny + 1) { fbc = -fbc; db = -db; fix = true; }
            }
            const Carry fwd = slope_fwd<+1>(cj1.E, cj2.E, cj1.V, cj2.V, cj1.U, cj2.U, fbc, fbr, K.udy, K);
            slope_rest<+1, FAST, REC>(cj.E, cj1.E, cj2.E, cj.V, cj2.V, cj.U, cj2.U, Hnj, Hnj1, fix, fix, dfb, db, K.udy,
                                      K, fbr, kOutLanes, ycar, fwd, Vyn, Uyn, Sn, dlon, dhin, okyn, &ycn);
            ycar = fwd;
        }
        float gnx, gny, gnz;
        {
            float a, b, c;
            face<FAST, REC>(okyj && okyn && !dryj && !dryj1, cj.E, cj.V, cj.U, Vyj, Uyj, dhij, cj1.E, cj1.V, cj1.U,
                            Vyn, Uyn, dlon, K, a, b, c, &gcn);
            gnx = a; gny = c; gnz = b;
        }
        // ---- branch record of row j (an interior row) ----
        if (REC && rec_lane) {
            rec_store(j, cj.U, cj.V);
            uint32_t code = 0u;
            if (C >= 1 && C <= nx + 2) {
                st(plane(A.tape_t), ocl, rj, T);
                code |= xc << kCodeX;
                if (C <= nx + 1) code |= fce << kCodeFx;
            }
            if (col_in) {
                st(plane(A.tape_s), ocl, rj, Sj);
                code |= (ycj << kCodeY) | (gcn << kCodeFy);
            }
            rec_code(j, code);
        }
        // ---- west face from the left lane ----
        const float fwx = from_left(fex), fwy = from_left(fey), fwz = from_left(fez);

        // ---- sources, RK update, store (:802-1004) ----
        if (store_lane) {
            const float Hm = cj.Hm4;
            const float ec = cj.E, uc = cj.U, vc = cj.V;
            const float hreg = ec + Hm;
            const float fd0 = div_k<FAST>(fex - fwx, K.dx, K.r_dx, K.l_dx) + div_k<FAST>(gnx - gsx, K.dy, K.r_dy, K.l_dy);
            const float fd1 = div_k<FAST>(fey - fwy, K.dx, K.r_dx, K.l_dx) + div_k<FAST>(gny - gsy, K.dy, K.r_dy, K.l_dy);
            const float fd2 = div_k<FAST>(fez - fwz, K.dx, K.r_dx, K.l_dx) + div_k<FAST>(gnz - gsz, K.dy, K.r_dy, K.l_dy);
            // wind, Coriolis and bottom slope of a wet cell.  The halves of
            // the means and depth differences are exact: 0.5 (w + e) + Hm is
            // one fma, and (g m) (0.5 D) = (0.5 g m) D
            auto sources = [&](float hu, float hv, float& st1, float& st2) {
                float X = A.wind_x, Y = A.wind_y;
                if (wgrid) wind_grid_value(wcell, A.wind_t, X, Y);
                const float eta_we = (ec - T) + (ec + T);
                const float eta_sn = (ec + Sj) + (ec - Sj);
                const float b1 = (K.half_g * fmaf(0.5f, eta_we, Hm)) * (He2 - Hw2);
                const float b2 = (K.half_g * fmaf(0.5f, eta_sn, Hm)) * (Hnj - Hsj);
                const float hu_cor = fcor * hv;
                const float hv_cor = (-fcor) * hu;
                st1 = (X + hu_cor) + div_k<FAST>(b1, K.dx, K.r_dx, K.l_dx);
                st2 = (Y + hv_cor) + div_k<FAST>(b2, K.dy, K.r_dy, K.l_dy);
            };
            float hu, hv, st1, st2;
            if (!dryj && none(!(hreg > K.cutoff))) {
                // every writing lane wet: no selects
                hu = uc * hreg;
                hv = vc * hreg;
                sources(hu, hv, st1, st2);
            } else {
                hu = 0.0f; hv = 0.0f; st1 = 0.0f; st2 = 0.0f;
                if (hreg > K.cutoff) {
                    hu = uc * hreg;
                    hv = vc * hreg;
                }
                if (hreg >= K.cutoff && ec != kDryFlag) sources(hu, hv, st1, st2);
            }
            const float L1 = -fd0;
            const float L2 = -fd1 + st1;
            const float L3 = -fd2 + st2;
            float Cf = 0.0f;
            if (friction) {   // quadratic bottom friction (:884-900)
                const float h = hreg;
                if (h < K.desing) {
                    const float uu = desingularize(h, hu, K.desing);
                    const float vv = desingularize(h, hv, K.desing);
                    Cf = (dt * A.r) * desingularize(h, sqrtf(uu * uu + vv * vv), K.desing);
                } else {
                    const float uu = hu / h, vv = hv / h;
                    Cf = ((dt * A.r) * sqrtf(uu * uu + vv * vv)) / h;
                }
            }
            float ue, uu, uv;
            if (rk_order < 3) {
                if (rk_step == 0) {
                    ue = ec + dt * L1;
                    uu = hu + dt * L2;
                    uv = hv + dt * L3;
                    if (friction) {
                        uu = uu / (1.0f + Cf);
                        uv = uv / (1.0f + Cf);
                    }
                } else {
                    ue = 0.5f * (ea + (ec + dt * L1));
                    uu = 0.5f * (ha + (hu + dt * L2));
                    uv = 0.5f * (va + (hv + dt * L3));
                    if (friction) {
                        uu = uu / (1.0f + 0.5f * Cf);
                        uv = uv / (1.0f + 0.5f * Cf);
                    }
                }
            } else {
                if (rk_step == 0) {
                    ue = ec + dt * L1;
                    uu = hu + dt * L2;
                    uv = hv + dt * L3;
                } else if (rk_step == 1) {
                    ue = 0.75f * ea + 0.25f * (ec + dt * L1);
                    uu = 0.75f * ha + 0.25f * (hu + dt * L2);
                    uv = 0.75f * va + 0.25f * (hv + dt * L3);
                } else {
                    ue = (ea + 2.0f * (ec + dt * L1)) / 3.0f;
                    uu = (ha + 2.0f * (hu + dt * L2)) / 3.0f;
                    uv = (va + 2.0f * (hv + dt * L3)) / 3.0f;
                }
            }
            const float floor_e = -Hm + K.cutoff;
            const bool gone = ue + Hm <= K.cutoff;
            if (!none(gone)) {
                rare();
                ue = gone ? floor_e : ue;
                uu = gone ? 0.0f : uu;
                uv = gone ? 0.0f : uv;
            }
            ue = fmaxf(floor_e, ue);
            st(r_eo, ocl, rj, ue);
            st(r_uo, ocl, rj, uu);
            st(r_vo, ocl, rj, uv);
            // periodic ghost images of the output (cells within two rows /
            // columns of a periodic side)
            if (ghost_cols || (pNS && (j <= 3 || j >= ny))) {
                rare();
                int rows[3] = {j, -1, -1}, cols[3] = {C, -1, -1};
                int nr = 1, nc = 1;
                if (pNS) {
                    if (j + ny <= ny + 3) rows[nr++] = j + ny;
                    if (j - ny >= 0) rows[nr++] = j - ny;
                }
                if (pEW) {
                    if (C + nx <= nx + 3) cols[nc++] = C + nx;
                    if (C - nx >= 0) cols[nc++] = C - nx;
                }
                for (int a = 0; a < nr; ++a) {
                    for (int b = 0; b < nc; ++b) {
                        if (a == 0 && b == 0) continue;
                        const uint32_t ro = (uint32_t)rows[a] * rowb, co = (uint32_t)cols[b] * 4u;
                        st(r_eo, co, ro, ue); st(r_uo, co, ro, uu); st(r_vo, co, ro, uv);
                    }
                }
            }
        }

        // ---- slide the window one row north ----
        ycj = ycn;
        gsx = gnx; gsy = gny; gsz = gnz;
        cj = cj1; cj1 = cj2;
        dryj = dryj1; dryj1 = dryj2;
        Uyj = Uyn; Vyj = Vyn; Sj = Sn; dhij = dhin; okyj = okyn;
        hc2 = hc3; hn2 = hn3; pl2 = pl3;
        Hsj = Hnj; Hnj = Hnj1;
    }
    // the last strip of a column records ghost rows ny+2 (its y slope
    // centre) and ny+3 (interior columns)
    if (REC && j1 == ny + 2 && rec_lane && col_in) {
        rec_store(ny + 2, cj.U, cj.V);
        st(plane(A.tape_s), ocl, (uint32_t)(ny + 2) * rowb, Sj);
        rec_code(ny + 2, ycj << kCodeY);
        rec_store(ny + 3, cj1.U, cj1.V);
        rec_code(ny + 3, 0u);
    }
}

}  // namespace march
}  // namespace gocean
