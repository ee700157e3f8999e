// mgr_radiation.hip -- radiation field: line emissivity/opacity along the
// traced ray pairs and the second-order Feautrier solve, fused in one kernel.
//
// Replaces Simulation::compute_radiation_field (src/Simulation/sim_radiation.tpp:56-338)
// with its inner calls Simulation::setup / get_eta_and_chi (simulation.tpp:185-481),
// Radiation::rescale_I_bdy (radiation.tpp:341-373), RayPair::solve
// (raypair_solver.tpp:200-388, n_off_diag 0 or 1: the same diagonal operator)
// and RayPair::update_Lambda (raypair_lambda.tpp:94-149); with scattering it
// also keeps each pair's u (Radiation::u, sim_radiation.tpp:226-262).  The
// image kernels (Simulation::compute_and_write_image) run the same elimination
// along a rest-frame trace.
//
// Work mapping (CDNA4, 64-wide wavefronts): one wavefront per origin cell and
// chunk of 64 frequency bins (lane = bin).  The wave loops over the nrays/2 ray
// pairs of its origin.  For every pair it lays out, from the cached traced
// steps, the points that can lie in a line window (lane = step, then lane =
// point; the spans of sub-points in the window are precomputed with the
// trace), brings their line rows (1/width and the emissivity/opacity
// prefactors per line) into LDS and walks them (sweep_pair).  Some FP32 models
// (many lines or bins, dark boundaries, very long steps) have the steps staged for
// a workgroup of several chunks instead (sweep_staged, per_point).  J and the Lambda*
// diagonal accumulate in FP64 registers over rays and are written once per
// (cell, bin): no atomics.  Workgroups are mapped to XCDs in contiguous origin
// ranges so that neighbouring origins share an L2.
//
// Bound: vector-instruction issue.  On the 64^3 envelope (48 rays, 186 bins) the
// FP32 kernel issues 2.0e10 vector instructions in 32 ms, 1.0 of one
// non-transcendental instruction per CU and cycle, of which the points' profiles
// and recurrences are 19.5 per point and wave, 65 % of all.  Decoding each
// step in the elimination loop and stepping every point took 49 ms; on the
// stress envelope (36^3, ~10 points per step) 44 against 19 ms.  FP64: 221
// against 152 ms and 192 against 97 ms.
//
// The tridiagonal Feautrier system of a ray pair is solved two-sided: each ray
// of the pair is eliminated from its boundary inwards in the Rybicki-Hummer
// (1+F) form and both eliminations meet at the origin, which yields u and the
// diagonal of the inverse there without storing or back-substituting the pair.
// With a = Dtau_{n-1}, b = Dtau_n the reference's F and Su recurrences, divided
// through by C_n, read F_n = (a+b) b/2 + (b/a) F_{n-1}/(1+F_{n-1}) and
// Z_n = (S_n (a+b) b/2 + (b/a) Z_{n-1}) / (1+F_n).  In the variables
// phi_n = F_n / b and zeta_n = Z_n / b every 1/a cancels:
//   h = (a+b)/2,  phi_n = h + phi_{n-1} q_{n-1},  q_n = 1/(1 + b phi_n),
//   zeta_n = (S_n h + zeta_{n-1}) q_n,
// one reciprocal per point.  The virtual start phi = q = 1, zeta = I_bdy, a = 0
// reproduces the boundary row F_0 = b(1 + b/2), Z_0 = (S b^2/2 + I b)/(1+F_0).
// At the origin, with h_o = (b_A + b_B)/2,
//   u = (S h_o + zeta_A + zeta_B) / (h_o + phi_A q_A + phi_B q_B),
//   Lambda = h_o / (h_o + phi_A q_A + phi_B q_B),
// and an empty side (origin on the boundary, incoming I_bdy of the origin's
// boundary cell) enters as the virtual start: phi q = 1, zeta = I, b = 0.
// phi stays below 1 + tau and q in (0, 1], so the FP32 variant neither
// overflows nor loses the optically thin limit.
// The kernels carry these in scaled variables, c = b/sqrt2, x = sqrt2 phi,
// z = sqrt2 zeta, y = x q + c and p = S c_prev + z_prev, in which
//   x_n = c_n + y_{n-1},  q_n = 1/(1 + c_n x_n),  y_n = x_n q_n + c_n,
//   z_n = (S_n c_n + p_n) q_n,
// so that no constant factor and no value from two points back is needed
// (no register copies around the loop); the virtual start is y = sqrt2,
// z = p = sqrt2 I, c = 0, and at the origin
//   u = (p_A + p_B) / (y_A + y_B),  Lambda = (c_A + c_B) / (y_A + y_B).
//
// Line profiles.  FP64 variant: the window of get_eta_and_chi is decided in
// FP64 exactly as the reference, or, where each bin meets one line, on the
// profile's argument (eta_chi_one).  FP32 variant: each lane evaluates the lines
// whose +-11-width window can contain its bin at any point of the model (its
// candidate lines; lines outside contribute exactly zero in FP64 too, and
// inside the window but beyond ~10 widths exp(-x^2) underflows FP32), with the
// offset x = ((nu_f - nu_l) + delta nu_f) / width formed from the per-lane
// difference nu_f - nu_l and the point's shift delta = shift - 1, which keeps
// the profile argument accurate in FP32.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <type_traits>
#include <vector>

#include "mgr_common.hpp"
#include "mgr_lds.hpp"
#include "mgr_ray.hpp"

using namespace mgr;

namespace {

constexpr int32_t ERR_NOT_BOUNDARY = 2;   // ray ends on a non-boundary cell
constexpr int32_t ERR_EMPTY_SIDE   = 4;   // empty ray at a non-boundary origin
constexpr int CH_MAX = 64;                // traced steps staged per chunk (at most)
constexpr int64_t WAVES_IN_FLIGHT = 8192;  // of the field kernels: 256 CUs, 8 waves per SIMD
constexpr int MAX_WAVES = 4;              // frequency chunks per workgroup

template <typename real> struct Prec;
template <> struct Prec<float> {
    using row_t = float4;   // (1/width, E, K, 0)
    static __device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
};
template <> struct Prec<double> {
    using row_t = double4;  // (11 width, 1/width, E, K)
    // the hardware reciprocal r (measured within 4.6e-8 of 1/x) times
    // 1/(1 - e) ~ 1 + e + e^2 of its residual e = 1 - x r: within an ulp (1.1e-16
    // measured), as two Newton steps, one instruction fewer.  The elimination's
    // arguments are normal numbers (chi scaled and 1 + c x >= 1).
    static __device__ __forceinline__ double rcp(double x)
    {
        const double r = __builtin_amdgcn_rcp(x);
        const double e = __builtin_fma(-x, r, 1.0);
        return __builtin_fma(r, __builtin_fma(e, e, e), r);
    }
};

// One traced step in LDS.  Sub-point m = 1..n of the step lies at shift s0 + m ds
// with path-length factor dz = dZ HDZ_SCALE and belongs to the current cell for
// m < half, to `cell` otherwise.  FP32 image kernel: Step; FP32 field kernel of
// staged steps: Step32, whose s0 is shift - 1.
struct alignas(32) Step {
    double  s0, ds, dz;
    int32_t nh;           // n | half << 14 (STEP_*)
    int32_t cell;
};
struct alignas(32) Step32 {
    float   s0, ds, dz;
    int32_t nh;           // n | half << 14 | out-of-window bits << 27: one 16-byte read with the above
    int32_t cell;
};

template <typename real>
struct RFArgs {
    int64_t N;
    int     F, L, nchunk, nwg, ngroups, grid_real, ch;
    int     pair_stride;                      // every pair_stride-th ray pair, weights times pair_stride
    int32_t o_begin;                          // first origin of this launch
    size_t  row_offset;                       // byte offset of the row region in LDS
    const LineTables *tb;
    const double  *nu;                        // [N*F]
    const typename Prec<real>::row_t *rows;   // [N*L]
    const int64_t *seg_off;
    const int32_t *nseg, *npts, *seg_cell;
    const double  *seg_shift, *seg_dZ;
    const int4    *seg_f32;                   // FP32 split of every step (cell, n | half << 14, s0, ds)
    const float   *seg_hdz32;                 // its dZ * HDZ_SCALE
    const int32_t *far_cell;                  // last emitted point of each (origin, ray), -1: none
    const double  *far_shift;
    const float   *far32;                     // cached far-end intensities [q F + f] of the FP32 kernel (or null)
    const double  *far64;                     // the same for the FP64 kernel (or null)
    uint64_t       L_magic;                   // ceil(2^32 / L): idx / L = (idx * L_magic) >> 32
    const double  *origin_shift;              // FP64 shift of the origin per entry (null: 1, co-moving)
    const uint8_t *step_mask;                 // per step, out-of-window bit per 64-bin chunk (or null)
    const uint16_t *span;                     // per chunk and step, the sub-points in the window (SPAN_*; or null)
    int64_t        span_stride;               // steps of a chunk
    const float   *near_p;                    // FP32: [L + 1] the spans' bound on p per line, and for bins of several lines
    const int32_t *near_bad;                  // FP32: set when a population exceeds the bounds behind the spans
    float          noop_lo, noop_hi;          // y in (noop_lo, noop_hi): a run's inner points change nothing
    bool           root_major;                // lane order (lane_bin)
    const int32_t *cell2bdy, *antipod;        // antipod: global ray indices
    const int32_t *cell_model;                // [N] model of each cell
    const int64_t *cell_qbase;                // [N] first (origin, ray) entry of the cell
    const int32_t *m_R, *m_rbase, *m_active;  // per model: rays, first global ray, still iterating
    const double  *I_bdy;                     // [NB*F]
    const double  *ray_w, *dshift_max;
    double         cand_lo, cand_hi;          // candidate-line bounds (FP32 variant)
    double         lstart_threshold;          // first line that can be in a window (FP64 variant)
    double        *J, *Lam;                   // [N*F]
    // RayPair::update_Lambda's sums: back-map of bin f to transition f_k[f]
    // (L: none) and root f_z[f], with the line data and profile widths
    const int32_t *f_k, *f_z;
    const double  *qw, *A_k, *freq_k, *pw;
    double        *Lpart;                     // [N][nchunk][L] one sum per wave and transition
    double        *u_out;                     // [R/2][N*F] per-pair u (scattering), or null
    int32_t       *err_flag;
    int            nband;                     // Lambda* bands (n_off_diag - 1) of k_lambda_band
    int64_t        band_S;                    // band slots per origin
    double        *band_part;                 // [N][nchunk][band_S][L]
    size_t         line_offset;               // FP64: byte offset of the line-frequency copy in LDS
    int            wave_lds;                  // field kernel: bytes of LDS of each wave
};

// ---- line profiles ----------------------------------------------------------

// exp(-t) for t >= 0: reduced by multiples of ln 2, whose double is taken in
// two parts, to |r| <= ln 2 / 2, and there the polynomial of degree 11 that
// meets exp at the 12 Chebyshev nodes of that interval (relative error below
// 1.7e-17), scaled by ldexp; 0 from t = 745.2 up to 1e40, where the polynomial
// overflows, and NaN for NaN.  18 instructions, without the range and sign
// handling of the library's exp.
constexpr double EXP_NEG_END = 746.0;   // 0 from here on
__device__ __forceinline__ double exp_neg_parts(double t, double &n)
{
    n = __builtin_rint(t * -1.4426950408889634);
    // ln 2 = 0x1.62e42fee00000p-1 (n times it is exact) + 1.9082149292705877e-10
    const double r = __builtin_fma(n, -1.9082149292705877e-10, __builtin_fma(n, -0x1.62e42fee00000p-1, -t));
    double p = 2.511003761756205e-08;
    p = __builtin_fma(p, r, 2.763263965412376e-07);
    p = __builtin_fma(p, r, 2.7557240918547625e-06);
    p = __builtin_fma(p, r, 2.480148548228773e-05);
    p = __builtin_fma(p, r, 0.00019841269890047143);
    p = __builtin_fma(p, r, 0.0013888888952314812);
    p = __builtin_fma(p, r, 0.008333333333319601);
    p = __builtin_fma(p, r, 0.04166666666648809);
    p = __builtin_fma(p, r, 0.1666666666666668);
    p = __builtin_fma(p, r, 0.5000000000000019);
    p = __builtin_fma(p, r, 1.0);
    return __builtin_fma(p, r, 1.0);
}

// From t = 1.5e9 on an int does not hold n: the instruction gives the nearest
// one, where a conversion in C++ is undefined.
__device__ __forceinline__ int nearest_int(double x)
{
    int i;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(i) : "v"(x));
    return i;
}
__device__ __forceinline__ double exp_neg(double t)
{
    double n;
    const double p = exp_neg_parts(t, n);
    return __builtin_ldexp(p, nearest_int(n));
}

// 0 where `in` is false, which it is to be beyond EXP_NEG_END.
__device__ __forceinline__ double exp_neg(double t, bool in)
{
    double n;
    const double p = exp_neg_parts(t, n);
    return __builtin_ldexp(p, in ? (int)n : -4000);
}

// FP64: get_eta_and_chi (simulation.tpp:385-481) for one lane with the exact
// window: skip while freq_diff > 11 width, include while freq_diff >= -11 width.
// row: the first line's row, the others `stride` apart.
__device__ __forceinline__ void eta_chi64(const RFArgs<double> &a, const double4 *__restrict__ row, int stride,
                                          const double *__restrict__ line, double fs, int lstart, double &eta,
                                          double &chi)
{
#pragma clang fp contract(off)
    // line[left lines from the last] runs with its row
    int left = a.L - 1 - lstart;
    line += lstart;
    row += lstart * stride;
    double fd = fs - *line;
    double4 v = *row;
    while (fd > v.x && left > 0) {
        left--;
        fd = fs - *++line;
        v = *(row += stride);
    }
    double e_acc = 0.0, c_acc = CHI_FLOOR * CHI_SCALE;
    while (fd >= -v.x) {
        const double x = fd * v.y;
        const double g = fs * exp_neg(x * x);   // the last line's window has no upper end
        e_acc += v.z * g;
        c_acc += v.w * g;
        if (left <= 0) break;
        left--;
        fd = fs - *++line;
        v = *(row += stride);
    }
    eta = e_acc;
    chi = c_acc;
}

// FP32: the lane's candidate lines la .. la+nc-1.  The first candidate is
// evaluated unconditionally (a lane without candidates carries an offset so
// large that its term is exactly zero); further candidates behind
// wave-uniform flags.  Rows hold 1/width scaled by sqrt(log2 e), so
// exp(-x^2) = exp2(-x'^2).
struct Lane32 {
    float  nuf;        // nu_f
    float  A0, A1;     // nu_f - nu_l of the first two candidates (or 1e30)
    int    la, l1, nc; // the first two (or any line), and how many
    bool   has2, has3; // wave-uniform: some lane has 2 / more than 2 candidates
    double nu_f64;
    double A0d, A1d;   // the same offsets in FP64 (FP32 image variant)
    const double *line;   // line frequencies (a copy in LDS in the field kernel)
};

// rows: the first line's row, the others `stride` apart; the shift - 1 is their w,
// or `delta` (GIVEN).
template <bool GIVEN = false>
__device__ __forceinline__ void eta_chi32(const RFArgs<float> &a, const Lane32 &ln, const float4 *__restrict__ rows,
                                          int stride, float &eta, float &chi, float delta = 0.0f)
{
#pragma clang fp contract(off)
    const float4 v0 = rows[ln.la * stride];
    if constexpr (!GIVEN) delta = v0.w;
    // nu_f (1 + delta) and (nu_f delta + nu_f - nu_l), each with one rounding
    const float nus = fmaf(delta, ln.nuf, ln.nuf);
    const float x0 = fmaf(delta, ln.nuf, ln.A0) * v0.x;
    const float g0 = nus * __builtin_amdgcn_exp2f(-(x0 * x0));
    float e_acc = v0.y * g0;
    float c_acc = fmaf(v0.z, g0, (float)(CHI_FLOOR * CHI_SCALE));
    if (ln.has2) {
        const float4 v1 = rows[ln.l1 * stride];
        const float x1 = fmaf(delta, ln.nuf, ln.A1) * v1.x;
        const float g1 = nus * __builtin_amdgcn_exp2f(-(x1 * x1));
        e_acc = fmaf(v1.y, g1, e_acc);
        c_acc = fmaf(v1.z, g1, c_acc);
        if (ln.has3) {
            for (int c = 2; c < ln.nc; c++) {
                const int l = ln.la + c;
                const float4 v = rows[l * stride];
                const float x = fmaf(delta, ln.nuf, (float)(ln.nu_f64 - ln.line[l])) * v.x;
                const float g = nus * __builtin_amdgcn_exp2f(-(x * x));
                e_acc = fmaf(v.y, g, e_acc);
                c_acc = fmaf(v.z, g, c_acc);
            }
        }
    }
    eta = e_acc;
    chi = c_acc;
}

// FP32 image variant: the shift s (absolute, FP64) and the offset from each
// candidate line in FP64, the profile and the sums in FP32.  An image bin can
// sit far out in a line's wing and meet the line only where the rest-frame
// shift cancels its offset; both terms are ~1e-4 nu there, and their FP32
// rounding (6e-12 nu) would be a visible fraction of a line width.
__device__ __forceinline__ void eta_chi32x(const RFArgs<float> &a, const float4 *__restrict__ row,
                                           const Lane32 &ln, double s, float &eta, float &chi)
{
    const double t = (s - 1.0) * ln.nu_f64;
    const float nus = (float)(t + ln.nu_f64);
    const float4 v0 = row[ln.la];
    const float x0 = (float)(t + ln.A0d) * v0.x;
    const float g0 = nus * __builtin_amdgcn_exp2f(-(x0 * x0));
    float e_acc = v0.y * g0;
    float c_acc = fmaf(v0.z, g0, (float)(CHI_FLOOR * CHI_SCALE));
    if (ln.has2) {
        const float4 v1 = row[ln.l1];
        const float x1 = (float)(t + ln.A1d) * v1.x;
        const float g1 = nus * __builtin_amdgcn_exp2f(-(x1 * x1));
        e_acc = fmaf(v1.y, g1, e_acc);
        c_acc = fmaf(v1.z, g1, c_acc);
        if (ln.has3) {
            for (int c = 2; c < ln.nc; c++) {
                const int l = ln.la + c;
                const float4 v = row[l];
                const float x = (float)(t + (ln.nu_f64 - a.tb->line[l])) * v.x;
                const float g = nus * __builtin_amdgcn_exp2f(-(x * x));
                e_acc = fmaf(v.y, g, e_acc);
                c_acc = fmaf(v.z, g, c_acc);
            }
        }
    }
    eta = e_acc;
    chi = c_acc;
}

// Radiation::rescale_I_bdy, scalar branch (radiation.tpp:341-373), at the
// count lo of the boundary cell's bins below the frequency (the grid is
// ascending, so that is the first bin >= freq, where search_with_notch from
// 0 stops): edge bins as they are, otherwise linear interpolation.
__device__ __forceinline__ double rescale_at(const double *__restrict__ nup, const double *__restrict__ Ib,
                                             int F, double fs, int lo)
{
#pragma clang fp contract(off)
    const int notch = lo < F ? lo : F - 1;
    if (notch == 0 || notch == F - 1) return Ib[notch];
    const double nu1 = nup[notch], nu2 = nup[notch - 1];
    const double I1 = Ib[notch], I2 = Ib[notch - 1];
    return (I2 - I1) / (nu2 - nu1) * (fs - nu1) + I1;
}

// The largest power of two <= F: the first step of the searches below.
__device__ __forceinline__ int search_top(int F) { return 1 << (31 - __builtin_clz((unsigned)F)); }

// Radiation::rescale_I_bdy of the boundary cell whose bins are nup (its
// intensities Ib) at frequency fs.  The count of bins below fs is found by
// halving steps from search_top(F): the same probes for every lane.
__device__ __forceinline__ double rescale_I_bdy(const double *__restrict__ nup,
                                                const double *__restrict__ Ib, int F, double fs)
{
    int lo = 0;
    for (int step = search_top(F); step > 0; step >>= 1)
        if (lo + step <= F && nup[lo + step - 1] < fs) lo += step;
    return rescale_at(nup, Ib, F, fs, lo);
}

// ---- Feautrier elimination state of one side ----------------------------------

__device__ __forceinline__ float fmad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmad(double a, double b, double c) { return __builtin_fma(a, b, c); }

// The recurrences are written with explicit fused multiply-adds (and
// contraction off), so that their rounding does not depend on how the
// compiler schedules or unrolls the loops around them.
template <typename real>
struct Sweep {
    real S_q, chi_q, hdz_q, cq;   // pending (outer) point: S, chi, its dz' and chi dz'
    real c, y, z, p, q;           // last closed interval and the scaled state, q = 1 / (1 + F) of the closed row

    // Virtual start.  With hdz_q = cq = 0 a step closes nothing: c = 0,
    // x = y, q = 1 exactly, so the first point may be stepped like any other.
    __device__ __forceinline__ void init(real I_far)
    {
        S_q = chi_q = hdz_q = cq = 0;
        c = 0;
        y = (real)SQRT2;
        z = (real)SQRT2 * I_far;
        p = z;
    }

    __device__ __forceinline__ void pend(real S, real chi, real hdz)
    {
#pragma clang fp contract(off)
        p = fmad(S, c, z);
        S_q = S;
        chi_q = chi;
        hdz_q = hdz;
        cq = chi * hdz;
    }

    // close the pending row with the next point (S, chi) inwards; the
    // interval takes the pending point's dz'
    __device__ __forceinline__ void step(real chi)
    {
#pragma clang fp contract(off)
        c = fmad(chi, hdz_q, cq);
        close_row();
    }

    // outward sweeps: the interval takes the new (outer) point's dz'
    __device__ __forceinline__ void step_out(real chi, real hdz)
    {
#pragma clang fp contract(off)
        c = (chi_q + chi) * hdz;
        close_row();
    }

    __device__ __forceinline__ void close_row()
    {
#pragma clang fp contract(off)
        const real x = c + y;
        q = Prec<real>::rcp(fmad(c, x, (real)1));
        y = fmad(x, q, c);
        z = fmad(S_q, c, p) * q;
    }
};

// ---- staging ----------------------------------------------------------------

// Stage the entries e = 0..cnt-1 of chunk [a, b): entry e holds step j = a-1+e
// (j = -1 is the origin) and the line rows of its cell.
template <typename S>
__device__ __forceinline__ void stage_chunk(const RFArgs<float> &a, int32_t o, int64_t q, int j0,
                                            int cnt, double dsm, S *__restrict__ st,
                                            float4 *__restrict__ rw)
{
    const int64_t s0 = a.seg_off[q];
    const int nthr = blockDim.x;
    for (int e = threadIdx.x; e < cnt; e += nthr) {
        const int j = j0 + e;
        S s;
        if (j < 0) {
            s.cell = o; s.nh = 0; s.s0 = 0; s.ds = 0; s.dz = 0;
        } else if constexpr (std::is_same_v<S, Step32>) {
            // split at trace time with the same FP64 arithmetic as below
            const int4 v = a.seg_f32[s0 + j];
            s.cell = v.x;
            s.nh = v.y | (a.step_mask ? (int)a.step_mask[s0 + j] << STEP_OUT_SHIFT : 0);
            s.s0 = __int_as_float(v.z);
            s.ds = __int_as_float(v.w);
            s.dz = a.seg_hdz32[s0 + j];
        } else {
            const int32_t c = a.seg_cell[s0 + j];
            const double sn = a.seg_shift[s0 + j];
            const double z = a.seg_dZ[s0 + j];
            const double sc = (j > 0) ? a.seg_shift[s0 + j - 1] : a.origin_shift[q];
            const StepSplit sp = split_step(sc, sn, z, dsm);
            s.cell = c;
            s.nh = sp.n | ((sp.interp ? sp.half : 0) << STEP_HALF_SHIFT);
            s.s0 = sp.interp ? sc : sn;               // absolute FP64 shift
            s.ds = sp.dshift;
            s.dz = sp.dZ * HDZ_SCALE;                 // dz'
        }
        st[e] = s;
    }
    __syncthreads();
    const int L = a.L;
    for (int idx = threadIdx.x; idx < cnt * L; idx += nthr) {
        // idx / L by a multiply with ceil(2^32 / L): exact for idx < 2^32 / L
        const int e = (int)(((uint64_t)(uint32_t)idx * a.L_magic) >> 32), l = idx - e * L;
        rw[idx] = a.rows[(int64_t)st[e].cell * L + l];
    }
    __syncthreads();
}

template <typename real>
struct LaneCtx;   // per-lane constants of the origin

template <>
struct LaneCtx<float> {
    Lane32 ln;
};
template <>
struct LaneCtx<double> {
    double nu_f;
    int    lstart;
    const double *line;   // line frequencies (a copy in LDS in the field kernel)
    double nu_l;          // frequency of the bin's only candidate line l (none: one far away)
    int    l;
    double top;           // upper end of that line's window (eta_chi_one)
};

template <typename real>
__device__ __forceinline__ void eval_point(const RFArgs<real> &a, const LaneCtx<real> &lc,
                                           const typename Prec<real>::row_t *__restrict__ row,
                                           real s, real &eta, real &chi);

template <>
__device__ __forceinline__ void eval_point<float>(const RFArgs<float> &a, const LaneCtx<float> &lc,
                                                  const float4 *__restrict__ row, float s,
                                                  float &eta, float &chi)
{
    // the rows' w is 0: the shift of the origin
    eta_chi32(a, lc.ln, row, 1, eta, chi);
}

template <>
__device__ __forceinline__ void eval_point<double>(const RFArgs<double> &a, const LaneCtx<double> &lc,
                                                   const double4 *__restrict__ row, double s,
                                                   double &eta, double &chi)
{
    double fs;
    {
#pragma clang fp contract(off)
        fs = s * lc.nu_f;
    }
    eta_chi64(a, row, 1, lc.line, fs, lc.lstart, eta, chi);
}

// shift of sub-point m: FP64 exactly s0 + m ds as Geometry::set_data;
// FP32 the offset shift - 1 in one fused multiply-add.
__device__ __forceinline__ double sub_point_shift(double s0, int m, double ds)
{
#pragma clang fp contract(off)
    return s0 + (double)m * ds;
}
__device__ __forceinline__ float sub_point_shift(float s0, int m, float ds)
{
    return fmaf((float)m, ds, s0);
}

__device__ __forceinline__ int rfl_int(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Incoming intensity at the far end of entry q (FP64, unscaled): the
// boundary intensity of the cell of the last emitted point, rescaled to that
// point's frequency shift * nu_f (Simulation::setup, simulation.tpp:266-272,
// 327-333); 0 for a ray without points.
template <typename real>
__device__ __forceinline__ double far_intensity(const RFArgs<real> &a, int64_t q, double nu_f, int F,
                                                int32_t &err)
{
    const int32_t cf = a.far_cell[q];
    if (cf < 0) return 0.0;
    const int32_t b = a.cell2bdy[cf];
    if (b < 0) {
        err |= ERR_NOT_BOUNDARY;
        return 0.0;
    }
    double fs;
    {
#pragma clang fp contract(off)
        fs = a.far_shift[q] * nu_f;
    }
    return rescale_I_bdy(a.nu + (int64_t)cf * F, a.I_bdy + (int64_t)b * F, F, fs);
}

// Scaled incoming intensity of entry q in the sweep's precision: the cache of
// that precision when it is built (the same value, computed once per trace,
// frequency grid and boundary intensities), else far_intensity.
template <typename real>
__device__ __forceinline__ real far_in(const RFArgs<real> &a, int64_t q, double nu_f, int F, int f, int32_t &err)
{
    if constexpr (sizeof(real) == 4) {
        if (a.far32) return a.far32[q * F + f];
    } else {
        if (a.far64) return a.far64[q * F + f];
    }
    return (real)(far_intensity(a, q, nu_f, F, err) * I_SCALE);
}

// The far-end intensity cache: one wave per (origin, ray) entry, its lanes
// over the bins, each the value far_in computes in the kernel of precision T
// (far_intensity with the entry's far cell, boundary and shift read once).
template <typename T>
__global__ __launch_bounds__(256) void k_far_cache(RFArgs<float> a, int Rmax, T *__restrict__ out,
                                                   int32_t *__restrict__ err_flag)
{
    const int F = a.F;
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const int64_t first = (int64_t)blockIdx.x * (blockDim.x / WAVE) + rfl_int((int)(threadIdx.x / WAVE));
    for (int64_t e = first; e < a.N * Rmax; e += (int64_t)gridDim.x * (blockDim.x / WAVE)) {
        const int32_t o = (int32_t)(e / Rmax);
        const int r = (int)(e - (int64_t)o * Rmax);
        if (r >= a.m_R[a.cell_model[o]]) continue;
        const int64_t q = a.cell_qbase[o] + r;
        T *dst = out + q * F;
        const int32_t cf = a.far_cell[q];
        const int32_t b = cf < 0 ? -1 : a.cell2bdy[cf];
        if (b < 0) {   // no points (0), or a far cell off the boundary (0 and an error)
            if (cf >= 0 && lane == 0) atomicOr(err_flag, ERR_NOT_BOUNDARY);
            for (int f = lane; f < F; f += WAVE) dst[f] = (T)(0.0 * I_SCALE);
            continue;
        }
        const double fsh = a.far_shift[q];
        const double *nup = a.nu + (int64_t)cf * F;
        const double *Ib = a.I_bdy + (int64_t)b * F;
        const double *nuo = a.nu + (int64_t)o * F;
        for (int f = lane; f < F; f += WAVE) {
            double fs;
            {
#pragma clang fp contract(off)
                fs = fsh * nuo[f];
            }
            dst[f] = (T)(rescale_I_bdy(nup, Ib, F, fs) * I_SCALE);
        }
    }
}

// One ray of an image pair, eliminated from its boundary end (incoming intensity
// I_far, scaled) inwards to the origin, which it leaves pending.
__device__ __forceinline__ Sweep<float> sweep_side(const RFArgs<float> &a, const LaneCtx<float> &lc,
                                                  int32_t o, int64_t q, float I_far, float S_o,
                                                  float chi_o, double dsm,
                                                  Step *__restrict__ st,
                                                  float4 *__restrict__ rw)
{
    Sweep<float> sw;
    sw.init(I_far);
    const int ns = a.nseg[q];
    const int L = a.L;
    const int CH = a.ch;
    for (int b_ = ns; b_ > 0; b_ -= CH) {
        const int a_ = b_ > CH ? b_ - CH : 0;
        const int cnt = b_ - a_ + 1;
        __syncthreads();   // the previous chunk is consumed by every wave
        stage_chunk(a, o, q, a_ - 1, cnt, dsm, st, rw);
        for (int e = cnt - 1; e >= 1; --e) {
            const int nh = rfl_int(st[e].nh);   // one readfirstlane: n and half are wave-uniform
            const int n = nh & STEP_N_MASK;
            const int half = (nh >> STEP_HALF_SHIFT) & STEP_HALF_MASK;
            const double s0 = st[e].s0, ds = st[e].ds;
            const float hdz = (float)st[e].dz;
            // sub-points m >= half lie in the step's cell (row e), m < half in
            // the previous one (row e-1); two loops keep each row's address
            // loop-invariant
            const float4 *rn = rw + e * L;
            const float4 *rc = rw + (e - 1) * L;
            const int mlo = half > 1 ? half : 1;
            for (int m = n; m >= mlo; --m) {
                float eta, chi;
                eta_chi32x(a, rn, lc.ln, sub_point_shift(s0, m, ds), eta, chi);
                const float S = eta * Prec<float>::rcp(chi);
                sw.step(chi);   // on the first point an exact no-op (c = 0, q = 1)
                sw.pend(S, chi, hdz);
            }
            for (int m = (half - 1 < n ? half - 1 : n); m >= 1; --m) {
                float eta, chi;
                eta_chi32x(a, rc, lc.ln, sub_point_shift(s0, m, ds), eta, chi);
                const float S = eta * Prec<float>::rcp(chi);
                sw.step(chi);
                sw.pend(S, chi, hdz);
            }
        }
    }
    sw.step(chi_o);   // the origin closes the innermost row and is left pending
    sw.pend(S_o, chi_o, (float)0);
    return sw;
}

// Continues an elimination outwards along entry q, from the origin (the
// pending point of sw) to the far end of the ray.  Each point closes the
// pending row with its own dZ (the outer point's, as Simulation::setup pairs
// them, simulation.tpp:306) and becomes the pending point; on return the
// far-end point is pending.
__device__ __forceinline__ void sweep_outward(const RFArgs<float> &a, const LaneCtx<float> &lc, int32_t o,
                                              int64_t q, double dsm, Sweep<float> &sw,
                                              Step *__restrict__ st,
                                              float4 *__restrict__ rw)
{
    const int ns = a.nseg[q];
    const int L = a.L;
    const int CH = a.ch;
    for (int a_ = 0; a_ < ns; a_ += CH) {
        const int b_ = a_ + CH < ns ? a_ + CH : ns;
        const int cnt = b_ - a_ + 1;
        __syncthreads();   // the previous chunk is consumed by every wave
        stage_chunk(a, o, q, a_ - 1, cnt, dsm, st, rw);
        for (int e = 1; e < cnt; ++e) {
            const int nh = rfl_int(st[e].nh);   // one readfirstlane: n and half are wave-uniform
            const int n = nh & STEP_N_MASK;
            const int half = (nh >> STEP_HALF_SHIFT) & STEP_HALF_MASK;
            const double s0 = st[e].s0, ds = st[e].ds;
            const float hdz = (float)st[e].dz;
            const float4 *rn = rw + e * L;
            const float4 *rc = rw + (e - 1) * L;
            const int mhi = half - 1 < n ? half - 1 : n;
            for (int m = 1; m <= mhi; ++m) {
                float eta, chi;
                eta_chi32x(a, rc, lc.ln, sub_point_shift(s0, m, ds), eta, chi);
                const float S = eta * Prec<float>::rcp(chi);
                sw.step_out(chi, hdz);
                sw.pend(S, chi, hdz);
            }
            for (int m = half > 1 ? half : 1; m <= n; ++m) {
                float eta, chi;
                eta_chi32x(a, rn, lc.ln, sub_point_shift(s0, m, ds), eta, chi);
                const float S = eta * Prec<float>::rcp(chi);
                sw.step_out(chi, hdz);
                sw.pend(S, chi, hdz);
            }
        }
    }
}

// u at the pending end point of a full sweep, closed by the incoming
// intensity I (scaled) there: the boundary row of RayPair::solve's last point
// in the elimination variables.
template <typename real>
__device__ __forceinline__ real end_u(const Sweep<real> &sw, real I)
{
    return (sw.p + (real)SQRT2 * I) * Prec<real>::rcp(sw.y + (real)SQRT2);
}

// FP64 with one candidate line per bin: get_eta_and_chi's window holds at most
// that line, x widths away: -11 <= x <= 11, or any x >= -11 of the last of all
// lines, which the reference's search never passes (top = EXP_NEG_END).  Beyond,
// eta is exactly 0, and so is J behind a dark boundary.  v: (anything, 1/width,
// E, K) of the line.
__device__ __forceinline__ void eta_chi_one(const LaneCtx<double> &lc, const double4 v, double s, double &eta,
                                            double &chi)
{
#pragma clang fp contract(off)
    const double fs = s * lc.nu_f;
    const double x = (fs - lc.nu_l) * v.y;
    const double t = x * fabs(x);
    const double g = fs * exp_neg(fabs(t), t >= -LINE_WINDOW * LINE_WINDOW && t <= lc.top);
    eta = v.z * g;
    chi = __builtin_fma(v.w, g, CHI_FLOOR * CHI_SCALE);
}

// Per-lane constants of origin o's bin and its own emissivity and opacity at
// the unshifted frequency nu_f (Simulation::setup takes the origin at
// nu(o, f), simulation.tpp:209-222).  ONE: no bin has more than one candidate
// line (known on the host), so the second-line code is compiled out.
template <typename real, bool X64 = false, bool ONE = false>
__device__ __forceinline__ void origin_point(const RFArgs<real> &a, double nu_f,
                                             const typename Prec<real>::row_t *__restrict__ orow,
                                             LaneCtx<real> &lc, real &S_o, real &chi_o)
{
    real eta_o;
    if constexpr (sizeof(real) == 4) {
        // candidate lines: nu_l (1 - w) <= s_max nu_f and nu_l (1 + w) >= s_min nu_f
        int la = 0;
        while (la < a.L && a.tb->line[la] * a.cand_lo < nu_f) la++;
        int lb = la;
        while (lb < a.L && a.tb->line[lb] * a.cand_hi <= nu_f) lb++;
        const int nc = lb - la;
        const int l0 = la < a.L ? la : a.L - 1;
        const int l1 = la + 1 < a.L ? la + 1 : a.L - 1;
        lc.ln.la = l0;
        lc.ln.nc = nc;
        lc.ln.nuf = (float)nu_f;
        lc.ln.nu_f64 = nu_f;
        lc.ln.A0 = (nc > 0) ? (float)(nu_f - a.tb->line[l0]) : 1.0e30f;
        lc.ln.A1 = (nc > 1) ? (float)(nu_f - a.tb->line[l1]) : 1.0e30f;
        lc.ln.A0d = (nc > 0) ? nu_f - a.tb->line[l0] : 1.0e30;
        lc.ln.A1d = (nc > 1) ? nu_f - a.tb->line[l1] : 1.0e30;
        lc.ln.l1 = l1;
        lc.ln.has2 = ONE ? false : __any(nc > 1);
        lc.ln.has3 = ONE ? false : __any(nc > 2);
        if constexpr (X64) eta_chi32x(a, orow, lc.ln, 1.0, eta_o, chi_o);
        else eval_point<real>(a, lc, orow, (real)0, eta_o, chi_o);
    } else {
        int ls = 0;
        while (ls < a.L - 1 && a.tb->line[ls] * a.lstart_threshold < nu_f) ls++;
        lc.nu_f = nu_f;
        lc.lstart = ls;
        if constexpr (ONE) {
            // a bin below its line's reach at every point has none: 0.1 nu is thousands of widths
            const double line = a.tb->line[ls];
            const bool last = ls == a.L - 1;
            lc.nu_l = line * a.cand_hi <= nu_f && (last || line * a.cand_lo >= nu_f) ? line : 0.9 * nu_f;
            lc.top = last && lc.nu_l == line ? EXP_NEG_END : LINE_WINDOW * LINE_WINDOW;
            lc.l = ls;
        }
        if constexpr (ONE) eta_chi_one(lc, orow[ls], 1.0, eta_o, chi_o);
        else eval_point<real>(a, lc, orow, (real)1, eta_o, chi_o);
    }
    S_o = eta_o * Prec<real>::rcp(chi_o);
}

// ---- the radiation field's sweep ---------------------------------------------

// A wave's LDS for one window of up to W = a.ch points (Window, W <= 64):
//   rows   [L][W + 1] the line rows of each point's cell, with the point's
//          shift in their spare component: the sweep reads a point's row and
//          shift in one access at a compile-time distance from the last
//          point's; the odd stride spreads the lines over the banks;
//   hdz    [WAVE] path-length factors dz';
//   stage  [WAVE] the points' shifts and cells;
//   owner  [WAVE] the points' steps (lanes of the batch).
template <typename real> struct Stage;
template <> struct Stage<float> { float s; int32_t cell; };
template <> struct Stage<double> { double s; int32_t cell, pad; };
template <typename real>
struct Window {
    using row_t = typename Prec<real>::row_t;
    row_t       *rows;
    real        *hdz;
    Stage<real> *stage;
    int         *owner;
    static constexpr size_t fixed = WAVE * (sizeof(real) + sizeof(Stage<real>) + sizeof(int));   // bytes beside the rows
    static constexpr size_t bytes(int64_t L, int points) { return fixed + sizeof(row_t) * L * (points + 1); }
    __device__ __forceinline__ void place(unsigned char *smem)
    {
        hdz = reinterpret_cast<real *>(smem);
        stage = reinterpret_cast<Stage<real> *>(hdz + WAVE);
        owner = reinterpret_cast<int *>(stage + WAVE);
        rows = reinterpret_cast<row_t *>(owner + WAVE);
    }
};

constexpr int BATCH = WAVE - 1;   // steps per batch: one lane each, the last lane for the cell before them

__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ bool lane_of(uint64_t m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
// Inclusive sum and maximum over the lanes up to this one (DPP row shifts and broadcasts).
__device__ __forceinline__ int scan_add(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    return x;
}
__device__ __forceinline__ int scan_max(int x)   // of values >= 0
{
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false));
    return x;
}
__device__ __forceinline__ int from_lane(int x, int lane) { return __builtin_amdgcn_ds_bpermute(lane << 2, x); }
__device__ __forceinline__ float from_lane(float x, int lane)
{
    return __int_as_float(from_lane(__float_as_int(x), lane));
}
__device__ __forceinline__ double from_lane(double x, int lane)
{
    return __hiloint2double(from_lane(__double2hiint(x), lane), from_lane(__double2loint(x), lane));
}

// The kernel's arguments, read from the kernarg segment where they are used:
// kept in scalar registers over the whole ray loop they spill into vector
// lanes, and every restore is a vector instruction.
template <typename real>
__device__ __forceinline__ const __attribute__((address_space(4))) RFArgs<real> *kernel_args()
{
    auto p = (const __attribute__((address_space(4))) RFArgs<real> *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// Emissivity and opacity at point p of a window (W points per line).
template <typename real, bool ONE>
__device__ __forceinline__ void eval_window(const RFArgs<real> &a, const LaneCtx<real> &lc, const Window<real> &win,
                                            int p, int W, real &eta, real &chi)
{
    if constexpr (sizeof(real) == 4) {
        eta_chi32(a, lc.ln, win.rows + p, W + 1, eta, chi);
    } else if constexpr (ONE) {
        const double4 v = win.rows[lc.l * (W + 1) + p];
        eta_chi_one(lc, v, v.x, eta, chi);
    } else {
        double fs;
        {
#pragma clang fp contract(off)
            fs = win.stage[p].s * lc.nu_f;
        }
        eta_chi64(a, win.rows + p, W + 1, lc.line, fs, lc.lstart, eta, chi);
    }
}

// How a wave passes over runs of consecutive points out of the window (FP32).
// Of such a run only the first point (at the far side) and the last one are
// evaluated.  The points between them close their rows with
// c <= 2 X dz'_max, X bounding chi out of the window, and have source
// functions S <= Smax.  With c below half an ulp of y, c y below 2^-25 and
// S c below half an ulp of p each of them leaves x = y, q = 1, y as it was and
// z = p = the value of p after the first point: the same bits as stepping
// them.  y and p are tested on every lane (noop_lo, noop_hi, p_min); a wave
// whose state fails the test goes on without skipping what the test needed:
//   SPAN   sub-points beyond the narrow window (span): the lines add at most
//          NEAR_CHI of the floor there, X = floor (1 + NEAR_CHI), S as bounded
//          by near_p;
//   WIDE   steps beyond MASK_WINDOW widths (step_mask): profiles are 0,
//          X = floor, S = 0 and any p will do;
//   NONE   every point is evaluated.
// The FP64 kernel steps every point, but evaluates only those within
// MASK_WINDOW64 widths (SPAN, or the steps that have one: WIDE): beyond, eta = 0
// and chi is the floor exactly.
struct Runs {
    enum { SPAN = 0, WIDE = 1, NONE = 2 };
};

// The two rays of a pair, the antipode's (entry qa of ns_a steps) first: each
// is eliminated from its boundary end inwards to the origin, which closes its
// innermost row, and adds its y, p and c to y2, p2 and c2 (an empty ray adds
// none of them); the whole call belongs to one wave.
//
// The cached steps of both rays form one list, each ray from its far end
// inwards, taken up to BATCH steps at a time, one lane each: the rays of most
// pairs fit one batch, whose set-up is about as much work as a dozen points.
// The lanes read the steps' in-window spans first and then only what the steps
// to be evaluated need.  The points of those steps are laid out one per lane
// (scan of the steps' point counts, owner by a maximum scan), a window at a
// time, and their rows and shifts go to LDS.  The elimination then walks the
// window: two LDS reads and the recurrence per point, with no per-step
// control and no work for the inner points of out-of-window runs.
template <typename real, bool ONE>
__device__ __forceinline__ void sweep_pair(const RFArgs<real> &a, const LaneCtx<real> &lc, int32_t o, int64_t qa,
                                           int ns_a, int64_t qr, int ns_r, real I_a, real I_r, real S_o, real chi_o,
                                           double dsm, float p_min, int chunk, int mode, const Window<real> &win,
                                           real &y2, real &p2, real &c2)
{
    using row_t = typename Prec<real>::row_t;
    constexpr bool F32 = sizeof(real) == 4;
    constexpr bool INROW = F32 || ONE;   // the rows have a component to spare for the shift
    constexpr int UNROLL = F32 || ONE ? 2 : 1;
    Sweep<real> sw;
    sw.init(ns_a > 0 ? I_a : I_r);
    const real chi_floor = (real)(CHI_FLOOR * CHI_SCALE);
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const auto *ka = kernel_args<real>();
    const int L = ka->L, W = ka->ch;
    // step g of the list lies at far_a - g on the antipode's ray (g < ns_a), at far_r - g on the other
    const int T = ns_a + ns_r;
    const int64_t far_a = ka->seg_off[qa] + ns_a - 1, far_r = ka->seg_off[qr] + T - 1;
    // the origin closes the ray's innermost row
    auto finish = [&]() {
        sw.step(chi_o);
        sw.pend(S_o, chi_o, (real)0);
        y2 += sw.y;
        p2 += sw.p;
        c2 += sw.c;
    };
    int g0 = 0, skip = 0;   // next step, and how many of its outermost points are done (FP32, after a failed test)
    while (g0 < T) {
        // steps with points in the window and those without (outm)
        const int nb = T - g0 < BATCH ? T - g0 : BATCH;
        const int split = ns_a - g0;   // lane of the second ray's first step
        const int g = g0 + lane;
        const int64_t at = (g < ns_a ? far_a : far_r) - g;
        unsigned span = SPAN_ALL;
        if (lane < nb) {
            if (mode == Runs::SPAN) span = ka->span[ka->span_stride * chunk + at];
            else if (mode == Runs::WIDE) span = (ka->step_mask[at] >> chunk) & 1 ? SPAN_NONE : SPAN_ALL;
        }
        const uint64_t valid = (1ull << nb) - 1;   // nb <= 63
        const uint64_t outm = __ballot(span == SPAN_NONE) & valid;
        const bool both = split > 0 && split <= nb;   // the first ray ends in this batch
        const uint64_t second = both && split < WAVE ? 1ull << split : 0;   // lane of the second one's first step
        // steps to load: those with points in the window, the ends of the runs of
        // others (runs end with their ray), and the steps before them, whose
        // cells they also touch (the next lane's)
        const uint64_t ends = F32 ? outm & ~((outm << 1) & (outm >> 1) & ~second & ~(second >> 1)) : outm;
        const uint64_t needm = (valid & ~outm) | ends;
        const uint64_t loadm = needm | (needm << 1);
        int32_t cell = o;
        int nh = 0;
        real st_s0 = 0, st_ds = 0, st_hdz = 0;
        const bool inner = g == ns_a - 1 || g == T - 1;   // the origin lies before this step
        if (lane_of(loadm) && g < T) {
            if constexpr (F32) {
                const int4 v = ka->seg_f32[at];
                cell = v.x;
                nh = v.y;
                st_s0 = __int_as_float(v.z);
                st_ds = __int_as_float(v.w);
                st_hdz = ka->seg_hdz32[at];
            } else {
                cell = ka->seg_cell[at];
                const double sn = ka->seg_shift[at];
                const double sc = inner ? 1.0 : ka->seg_shift[at - 1];   // co-moving: the origin's shift is 1
                const StepSplit sp = split_step(sc, sn, ka->seg_dZ[at], dsm);
                nh = sp.n | ((sp.interp ? sp.half : 0) << STEP_HALF_SHIFT);
                st_s0 = sp.interp ? sc : sn;
                st_ds = sp.dshift;
                st_hdz = sp.dZ * HDZ_SCALE;
            }
        }
        const int32_t next = from_lane(cell, lane + 1);   // on every lane: an idle one would hand out nothing
        const int32_t before = inner ? o : next;
        // The sub-points of a step, from its far end inwards: n - hi out of the
        // window, then `in` inside it, then hi - in outside again (hi = in = 0: a
        // step of outm).
        const int n_all = nh & STEP_N_MASK, half = (nh >> STEP_HALF_SHIFT) & STEP_HALF_MASK;
        const int n = n_all - (lane == 0 ? skip : 0);
        const bool out = lane_of(outm);
        int hi = (((int)(span >> 8) + 1) * n_all + 255) >> 8;
        hi = out ? 0 : hi < n ? hi : n;
        const int in = out ? 0 : hi - (((int)(span & 255) * n_all) >> 8);
        // Of a run of out-of-window points only the first and the last are
        // evaluated (FP32).  A run at a ray's far end needs no first one:
        // nothing is pending yet, and c = 0 closes nothing.
        int cf, cn = hi > in ? 1 : 0;   // records before and after the points in the window
        bool first = false;             // the first record is the run's first point
        if constexpr (F32) {
            const uint64_t far_out = __ballot(out || n > hi) & valid, near_out = __ballot(out || hi > in) & valid;
            const uint64_t fresh = second | ((g0 == 0 || g0 == ns_a) && skip == 0 ? 1 : 0);
            // a run begins with this step's outer points, or ends with its inner ones
            const uint64_t begins = far_out & ~((near_out << 1) & ~second);
            const uint64_t stops = near_out & ~((far_out >> 1) & ~(second >> 1));
            first = lane_of(begins & ~fresh);
            const int outer = n - hi;   // points of the outer piece
            const bool closes = !out || lane_of(stops);   // the outer piece ends its run
            cf = outer > 0 ? (first ? 1 : 0) + (closes && !(first && outer == 1) ? 1 : 0) : 0;
            if (hi > in + 1 && lane_of(stops)) cn = 2;
        } else {
            cf = n > hi ? 1 : 0;   // one record for all of them
        }
        const int cnt = lane < nb ? cf + in + cn : 0;
        const int incl = scan_add(cnt);
        const int total = __builtin_amdgcn_readlane(incl, WAVE - 1);
        const int base = incl - cnt;
        const int turn = both ? __builtin_amdgcn_readlane(incl, split - 1) : INT32_MAX;   // points of the first ray
        bool pending = both;
        const int pack1 = n | hi << 14 | cf << 28 | (first ? 1 << 30 : 0);
        const int pack2 = in | half << 14;
        int before_window = 0;   // the last record's step and sub-point, of the window before
        bool again = false;
        for (int w0 = 0; w0 < total; w0 += W) {
            const int cw = total - w0 < W ? total - w0 : W;
            wave_lds_fence();   // the previous window is consumed
            if (F32 && w0 > 0) before_window = rfl_int(win.owner[W - 1]);
            wave_lds_fence();
            win.owner[lane] = 0;
            wave_lds_fence();
            // (base, lane) of the step that begins at a point, or before the window and ends in it
            if (cnt > 0 && base < w0 + W && base + cnt > w0) win.owner[base > w0 ? base - w0 : 0] = base << 6 | lane;
            wave_lds_fence();
            const int bl = scan_max(win.owner[lane]);
            const int own = bl & (WAVE - 1);
            const int p1 = from_lane(pack1, own), p2_ = from_lane(pack2, own);
            const int t = w0 + lane - (bl >> 6), k = t - ((p1 >> 28) & 3);
            const int o_hi = (p1 >> 14) & STEP_N_MASK, o_in = p2_ & STEP_N_MASK;
            const bool head = t == 0 && (p1 >> 30) & 1;
            const bool outer = k < 0, after = k > o_in;
            bool mark;
            int m = o_hi - k;
            if constexpr (F32) {
                mark = (outer && !head) || after;   // a run's last point
                if (outer) m = head ? p1 & STEP_N_MASK : o_hi + 1;
                if (after) m = 1;
            } else {
                mark = outer || k >= o_in;
            }
            Stage<real> sg;
            sg.s = sub_point_shift(from_lane(st_s0, own), m, from_lane(st_ds, own));
            const int32_t c_own = from_lane(cell, own), c_before = from_lane(before, own);
            sg.cell = m < ((p2_ >> 14) & STEP_HALF_MASK) ? c_before : c_own;
            if constexpr (!F32) {
                if (mark) sg.cell = outer ? (p1 & STEP_N_MASK) - o_hi : o_hi - o_in;   // its sub-points
            }
            uint64_t marks = __ballot(lane < cw && mark);
            win.hdz[lane] = from_lane(st_hdz, own);
            win.stage[lane] = sg;
            if constexpr (F32) win.owner[lane] = own << 14 | m;
            wave_lds_fence();
            {
                // the rows of WAVE / L points at a time, lane e L + l line l of point e
                const int per = WAVE / L;
                const int e0 = (int)(((uint64_t)(uint32_t)lane * ka->L_magic) >> 32), l = lane - e0 * L;
                const row_t *src = ka->rows + l;
                row_t *dst = win.rows + l * (W + 1);
                if (e0 < per)
                    for (int e = e0; e < cw; e += per) {
                        if (!F32 && ((marks >> e) & 1)) continue;
                        const Stage<real> sg_e = win.stage[e];
                        const row_t v = src[(uint32_t)sg_e.cell * (uint32_t)L];   // N L rows < 2^32
                        if constexpr (F32) dst[e] = make_float4(v.x, v.y, v.z, sg_e.s);
                        else dst[e] = make_double4(INROW ? sg_e.s : v.x, v.y, v.z, v.w);
                    }
            }
            wave_lds_fence();
            int p = 0;
            for (;;) {
                const int e = marks ? (int)__builtin_ctzll(marks) : cw;
                const bool turns = pending && turn - w0 <= e;
                const int stop = turns ? turn - w0 : e;
#pragma unroll UNROLL
                for (; p < stop; ++p) {
                    real eta, chi;
                    eval_window<real, ONE>(a, lc, win, p, W, eta, chi);
                    const real S = eta * Prec<real>::rcp(chi);
                    sw.step(chi);   // on a ray's first point an exact no-op (c = 0, q = 1)
                    sw.pend(S, chi, win.hdz[p]);
                }
                if (turns) {
                    finish();
                    sw.init(I_r);
                    pending = false;
                    continue;
                }
                if (e >= cw) break;
                if constexpr (F32) {
                    if (__all(sw.y > a.noop_lo && sw.y < a.noop_hi && sw.p > p_min)) {
                        float eta, chi;
                        eval_window<real, ONE>(a, lc, win, e, W, eta, chi);
                        const float h = win.hdz[e];
                        sw.z = sw.p;
                        sw.S_q = eta * Prec<real>::rcp(chi);
                        sw.hdz_q = h;
                        sw.cq = chi * h;
                    } else {
                        // go on in the next mode from the point after the last record, or
                        // from the ray's first point if this run begins the ray
                        if (w0 + e == turn) {
                            g0 = ns_a;
                            skip = 0;
                        } else if (w0 + e > 0) {
                            const int rec = e > 0 ? rfl_int(win.owner[e - 1]) : before_window;
                            const int m_done = rec & STEP_N_MASK;
                            g0 += rec >> 14;
                            skip = rfl_int(ka->seg_f32[(g0 < ns_a ? far_a : far_r) - g0].y & STEP_N_MASK) - (m_done - 1);
                            if (m_done == 1) {
                                g0++;
                                skip = 0;
                            }
                        }
                        mode++;
                        p_min = -FLT_MAX;
                        again = true;
                        break;
                    }
                } else {
                    // out of the window: eta = 0 and chi at the floor at each of its points
                    const real h = win.hdz[e];
                    for (int i = rfl_int(win.stage[e].cell); i >= 1; --i) {
                        sw.step(chi_floor);
                        sw.pend((real)0, chi_floor, h);
                    }
                }
                marks &= marks - 1;
                p = e + 1;
            }
            if (again) break;
        }
        if (!again) {
            g0 += nb;
            skip = 0;
        }
    }
    if (ns_r > 0) finish();
}

// One ray of a pair (entry q, which has points) by steps staged for the whole
// workgroup (FP32): eliminated from its boundary end inwards to the origin, which
// it leaves pending.  Out-of-window steps (step_mask) have eta = 0 and chi at the
// floor at every sub-point, which are stepped but not evaluated; while y passes the
// test (Runs) only the run's first one is.
__device__ __forceinline__ Sweep<float> sweep_staged(const RFArgs<float> &a, const LaneCtx<float> &lc, int32_t o,
                                                    int64_t q, float I_far, float S_o, float chi_o, int chunk,
                                                    Step32 *__restrict__ st, float4 *__restrict__ rw)
{
    Sweep<float> sw;
    sw.init(I_far);
    const float chi_floor = (float)(CHI_FLOOR * CHI_SCALE);
    // this wave's out-of-window bit in a staged nh word (none past the masked chunks)
    const unsigned cbit = chunk < STEP_MASK_CHUNKS ? 1u << (STEP_OUT_SHIFT + chunk) : 0u;
    const int L = a.L, CH = a.ch;
    auto uniform = [](float x) { return __int_as_float(rfl_int(__float_as_int(x))); };
    // s0 and ds stay in vector registers: one scalar operand per FMA
    auto read = [&](int e) { return reinterpret_cast<const float4 *>(st + e)[0]; };
    const int ns = rfl_int(a.nseg[q]);
    bool noop = false;   // y is in range since the run's first point
    for (int b_ = ns; b_ > 0; b_ -= CH) {
        const int a_ = b_ > CH ? b_ - CH : 0;
        const int cnt = b_ - a_ + 1;
        __syncthreads();   // the previous chunk is consumed by every wave
        stage_chunk(a, o, q, a_ - 1, cnt, 0.0, st, rw);
        int e = cnt - 1;
        while (e >= 1) {
            float4 v = read(e);
            int nh = rfl_int(__float_as_int(v.w));   // n, half and the bits are wave-uniform
            if (!((unsigned)nh & cbit)) {
                noop = false;
                // a run of steps with points inside a line window, in a loop of its
                // own so that the sweep state keeps its registers
                for (;;) {
                    const int n = nh & STEP_N_MASK;
                    __builtin_assume(n >= 1);   // a traced step emits 1 .. 10000 points
                    const int half = (nh >> STEP_HALF_SHIFT) & STEP_HALF_MASK;
                    const float hdz = uniform(v.z);
                    // sub-points m >= half lie in the step's cell (row e), m < half in
                    // the previous one (row e-1)
                    const float4 *rn = rw + e * L, *rc = rw + (e - 1) * L;
                    const int mlo = half > 1 ? half : 1;
                    for (int m = n; m >= mlo; --m) {
                        float eta, chi;
                        eta_chi32<true>(a, lc.ln, rn, 1, eta, chi, sub_point_shift(v.x, m, v.y));
                        sw.step(chi);   // on the first point an exact no-op (c = 0, q = 1)
                        const float S = eta * Prec<float>::rcp(chi);   // after the step: no copy of the last one
                        sw.pend(S, chi, hdz);
                    }
                    for (int m = (half - 1 < n ? half - 1 : n); m >= 1; --m) {
                        float eta, chi;
                        eta_chi32<true>(a, lc.ln, rc, 1, eta, chi, sub_point_shift(v.x, m, v.y));
                        sw.step(chi);
                        const float S = eta * Prec<float>::rcp(chi);
                        sw.pend(S, chi, hdz);
                    }
                    if (--e < 1) break;
                    v = read(e);
                    nh = rfl_int(__float_as_int(v.w));
                    if ((unsigned)nh & cbit) break;
                }
                if (e < 1) break;
            }
            // an out-of-window step: its first sub-point closes the row of the last evaluated point
            const int n = nh & STEP_N_MASK;
            __builtin_assume(n >= 1);
            const float hdz = uniform(v.z);
            if (!noop) {
                sw.step(chi_floor);
                sw.pend(0.0f, chi_floor, hdz);
                noop = __all(sw.y > a.noop_lo && sw.y < a.noop_hi);
                if (!noop) {
                    for (int m = n - 1; m >= 1; --m) {
                        sw.step(chi_floor);
                        sw.pend(0.0f, chi_floor, hdz);
                    }
                    --e;
                    continue;
                }
            }
            // pass over the out-of-window steps that follow in the chunk, keeping the last one's dz'
            int last = e;
            while (last > 1 && ((unsigned)rfl_int(st[last - 1].nh) & cbit)) last--;
            const float hdz_l = last == e ? hdz : uniform(st[last].dz);
            sw.hdz_q = hdz_l;
            sw.cq = chi_floor * hdz_l;
            e = last - 1;
        }
    }
    sw.step(chi_o);   // the origin closes the innermost row and is left pending
    sw.pend(S_o, chi_o, 0.0f);
    return sw;
}

// This wave's share of the Lambda* diagonal per transition
// (RayPair::update_Lambda, raypair_lambda.tpp:94-149, n_off_diag 0):
// Ls(p,k) = sum over the bins f of transition k of
// A_k w_z nu_f phi_k(nu_f) Lam(p,f), with Lam = sum_r 2 w_r L_diag / chi as
// the kernel accumulates it.  The wave sums its lanes' terms per transition
// in a fixed butterfly order and lane k writes transition k's sum;
// k_lambda_sum adds the waves of a cell in chunk order.
template <typename real>
__device__ __forceinline__ void lambda_partials(const RFArgs<real> &a, int32_t o, int chunk, bool active, int f,
                                                double nu_f, double lam_f)
{
    const int L = a.L;
    const int k = active ? a.f_k[f] : L;
    double term = 0.0;
    if (k < L) {
        const double freq_line = a.freq_k[k];
        const double iw = 1.0 / (freq_line * a.pw[(int64_t)a.tb->line_spec[k] * a.N + o]);   // the line's species
        const double x = iw * (nu_f - freq_line);
        const double prof = iw * INVERSE_SQRT_PI * (1.0 / exp(x * x));
        term = a.A_k[k] * a.qw[a.f_z[f]] * (nu_f * prof * lam_f);
    }
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    // transitions present in this wave: [kmin, kmax]
    int kmin = k, kmax = k < L ? k : -1;
    for (int off = WAVE / 2; off >= 1; off >>= 1) {
        kmin = min(kmin, __shfl_xor(kmin, off));
        kmax = max(kmax, __shfl_xor(kmax, off));
    }
    double mine = 0.0;
    for (int kk = kmin; kk <= kmax; kk++) {
        double v = (k == kk) ? term : 0.0;
        for (int off = WAVE / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off);
        v = __shfl(v, 0);   // lane 0's order for every lane
        if (lane == kk) mine = v;
    }
    if (chunk < a.nchunk && lane < L)
        a.Lpart[((int64_t)o * a.nchunk + chunk) * L + lane] = mine;
}

// One wave's bins of one origin: the pairs by sweep_pair, each wave with a window
// of its own, or by sweep_staged (STAGED).
template <typename real, bool ONE, bool STAGED>
__device__ __forceinline__ void field_of_origin(RFArgs<real> a)
{
    using row_t = typename Prec<real>::row_t;
    extern __shared__ __align__(16) unsigned char smem[];
    const int wave = rfl_int((int)(threadIdx.x / WAVE));
    Window<real> win;
    if constexpr (!STAGED) win.place(smem + wave * a.wave_lds);

    // XCD-aware order: consecutive workgroups go to different XCDs, so hand
    // each XCD a contiguous range of origins.
    const int G = gridDim.x;
    const int per = G >> 3;
    const int bid = blockIdx.x;
    const int logical = (bid & 7) * per + (bid >> 3);
    if (logical >= a.grid_real) return;   // whole workgroup: before any barrier
    const int32_t o = a.o_begin + (int32_t)(logical / a.ngroups);
    const int32_t mdl = a.cell_model[o];
    if (!a.m_active[mdl]) return;         // converged model of a batch: whole workgroup
    const int group = logical - (o - a.o_begin) * a.ngroups;
    const int chunk = rfl_int(group * a.nwg + wave);   // wave-uniform
    LaneCtx<real> lc;
    if constexpr (!ONE) {
        // the line frequencies that bins of several lines read at every point, in LDS
        double *lt = reinterpret_cast<double *>(smem + a.line_offset);
        for (int i = (int)threadIdx.x; i < a.L; i += (int)blockDim.x) lt[i] = a.tb->line[i];
        __syncthreads();
        if constexpr (sizeof(real) == 4) lc.ln.line = lt;
        else lc.line = lt;
    }
    if (!STAGED && chunk >= a.nchunk) return;   // a wave without bins: no barrier follows
    const int F = a.F;
    const int slot = chunk * WAVE + (int)(threadIdx.x & (WAVE - 1));
    const bool active = slot < F;
    const int f = lane_bin(active ? slot : F - 1, a.L, F, a.root_major);
    const double nu_f = a.nu[(int64_t)o * F + f];
    const double dsm = sizeof(real) == 8 ? a.dshift_max[o] : 0.0;
    const int32_t bo = a.cell2bdy[o];
    const row_t *orow = a.rows + (int64_t)o * a.L;

    real S_o, chi_o;
    origin_point<real, false, ONE>(a, nu_f, orow, lc, S_o, chi_o);
    // how out-of-window runs are passed over (Runs)
    int mode = Runs::NONE;
    float p_near = -FLT_MAX;
    if (!STAGED && chunk < STEP_MASK_CHUNKS) {
        if constexpr (sizeof(real) == 4) {
            if (a.step_mask) mode = Runs::WIDE;
            if (a.step_mask && a.span && *a.near_bad == 0) {
                mode = Runs::SPAN;
                p_near = lc.ln.nc > 1 ? a.near_p[a.L] : a.near_p[lc.ln.la];
            }
        } else if (a.step_mask) {
            mode = a.span ? Runs::SPAN : Runs::WIDE;
        }
    }
    mode = rfl_int(mode);

    int32_t err = 0;
    double J_acc = 0.0, Lam_acc = 0.0;
    const int rb = a.m_rbase[mdl];
    const int Rh = a.m_R[mdl] / 2;
    const int64_t qb = a.cell_qbase[o];
    const double wsc = 2.0 * (double)a.pair_stride;
    for (int r = 0; r < Rh; r += a.pair_stride) {
        const int ar = a.antipod[rb + r];
        const double w2 = wsc * a.ray_w[rb + r];
        const int64_t qr = qb + r;
        const int64_t qa = qb + (ar - rb);
        const int ns_r = rfl_int(a.nseg[qr]);   // a step has at least one point
        const int ns_a = rfl_int(a.nseg[qa]);
        if (ns_r == 0 && ns_a == 0) {
            // ndep == 1: u = I_bdy of the origin's boundary entry (sim_radiation.tpp:243-264)
            if (bo < 0) { err |= ERR_EMPTY_SIDE; continue; }
            const double Ib = a.I_bdy[(int64_t)bo * F + f];
            J_acc += w2 * Ib;
            if (a.u_out && active) a.u_out[((int64_t)r * a.N + o) * F + f] = Ib;
            continue;
        }
        // an empty ray (the origin is a boundary cell) is the virtual start with
        // I_bdy of the origin's boundary entry
        real y2 = 0, p2 = 0, c2 = 0, z_o = 0;
        if (ns_a == 0 || ns_r == 0) {
            if (bo < 0) err |= ERR_EMPTY_SIDE;
            else z_o = (real)SQRT2 * (real)(a.I_bdy[(int64_t)bo * F + f] * I_SCALE);
            y2 = (real)SQRT2;
        }
        if constexpr (STAGED) {
            Step32 *st = reinterpret_cast<Step32 *>(smem);
            float4 *rw = reinterpret_cast<float4 *>(smem + a.row_offset);
            // one call for both rays, the antipode's first
            for (int64_t q = ns_a > 0 ? qa : qr;; q = qr) {
                const float I = far_in<float>(a, q, nu_f, F, f, err);
                const Sweep<float> sw = sweep_staged(a, lc, o, q, I, S_o, chi_o, chunk, st, rw);
                y2 += sw.y;
                p2 += sw.p;
                c2 += sw.c;
                if (q == qr || ns_r == 0) break;
            }
        } else {
            const real I_a = ns_a > 0 ? far_in<real>(a, qa, nu_f, F, f, err) : (real)0;
            const real I_r = ns_r > 0 ? far_in<real>(a, qr, nu_f, F, f, err) : (real)0;
            sweep_pair<real, ONE>(a, lc, o, qa, ns_a, qr, ns_r, I_a, I_r, S_o, chi_o, dsm, p_near, chunk, mode, win,
                                  y2, p2, c2);
        }
        const real den = Prec<real>::rcp(y2);
        real u;
        {
#pragma clang fp contract(off)
            u = (p2 + z_o) * den;
        }
        const real lam = c2 * den;
        const double u64 = (double)u * (1.0 / I_SCALE);
        J_acc += w2 * u64;
        Lam_acc += w2 * (double)lam;
        if (a.u_out && active) a.u_out[((int64_t)r * a.N + o) * F + f] = u64;   // radiation.u[R][ind]
    }
    if (err) atomicOr(a.err_flag, err);
    const double lam_f = Lam_acc * CHI_SCALE / (double)chi_o;
    if (active) {
        a.J[(int64_t)o * F + f] = J_acc;
        a.Lam[(int64_t)o * F + f] = lam_f;
    }
    lambda_partials(a, o, chunk, active, f, nu_f, lam_f);
}

// FP32: at least 8 waves per SIMD (at most 64 VGPRs), which hide the LDS
// latency of the line rows; 6 where bins have several lines, whose second
// line's registers spill at 64; FP64: 4.  The waves of a workgroup
// share nothing but the line table.
template <typename real, bool ONE>
__global__ __launch_bounds__(WAVE * MAX_WAVES) __attribute__((amdgpu_waves_per_eu(sizeof(real) == 4 ? (ONE ? 8 : 6) : 4)))
void k_radiation_field(RFArgs<real> a)
{
    field_of_origin<real, ONE, false>(a);
}

// The same with steps and their line rows staged for the workgroup's waves, which
// is the faster way where a point's rows are many or few points are passed over
// (per_point).
template <bool ONE>
__global__ __launch_bounds__(WAVE * MAX_WAVES) __attribute__((amdgpu_waves_per_eu(8)))
void k_field_staged(RFArgs<float> a)
{
    field_of_origin<float, ONE, true>(a);
}

// The points of a ray pair in order: entry qx from its far end inwards, the
// origin, then entry qy outwards, at most ny points of it.  visit(t, eta, chi,
// h, p) gets the visit count t (uniform in the wave), the emissivity and opacity
// of the lane's bin there, the path factor h of the interval between the point and the one
// visited before it, which is that of the interval's outer point
// (Simulation::setup, simulation.tpp:233-240, 292-299; 0 for the first point),
// and the point's place p in the window (its shift and cell in win.stage).
//
// As in sweep_pair, up to WAVE steps of the pair lie on the lanes, and their
// points a window at a time, with the line rows of those inside the line
// window in LDS; at the others (by the spans, or by the steps' bits without them)
// eta = 0 and chi is the floor.
template <bool ONE, typename Visit>
__device__ __forceinline__ void walk_pair(const RFArgs<double> &a, const LaneCtx<double> &lc, int32_t o, int64_t qx,
                                          int64_t qy, int ny, double dsm, int chunk, const Window<double> &win,
                                          Visit &&visit)
{
    const int lane = (int)(threadIdx.x & (WAVE - 1));
    const auto *ka = kernel_args<double>();
    const int L = ka->L, W = ka->ch;
    const int nsx = rfl_int(ka->nseg[qx]), nsy = rfl_int(ka->nseg[qy]);
    const int T = nsx + 1 + (nsy < ny ? nsy : ny);   // steps; a step has at least one point
    int left = rfl_int(ka->npts[qx]) + 1 + ny;       // points
    const int64_t bx = ka->seg_off[qx], by = ka->seg_off[qy];
    const bool spans = ka->span && chunk < STEP_MASK_CHUNKS, bits = !spans && ka->step_mask && chunk < STEP_MASK_CHUNKS;
    int t = 0;
    double h_last = 0.0;   // path factor of the step before this batch
    for (int g0 = 0; g0 < T; g0 += WAVE) {
        const int g = g0 + lane;
        const bool inward = g < nsx, outward = g > nsx && g < T;
        const int j = inward ? nsx - 1 - g : g - nsx - 1;
        const int64_t at = (inward ? bx : by) + j;
        unsigned span = SPAN_ALL;
        int32_t c_next = o, c_prev = o;
        int n = g == nsx ? 1 : 0, half = 0;
        double s0 = 1.0, ds = 0.0, h = 0.0;
        if (inward || outward) {
            if (spans) span = ka->span[ka->span_stride * chunk + at];
            else if (bits) span = (ka->step_mask[at] >> chunk) & 1 ? SPAN_NONE : SPAN_ALL;
            c_next = ka->seg_cell[at];
            const double sn = ka->seg_shift[at];
            double sc = ka->origin_shift ? ka->origin_shift[inward ? qx : qy] : 1.0;   // co-moving: the origin's is 1
            if (j > 0) {
                c_prev = ka->seg_cell[at - 1];
                sc = ka->seg_shift[at - 1];
            }
            const StepSplit sp = split_step(sc, sn, ka->seg_dZ[at], dsm);
            n = sp.n;
            half = sp.interp ? sp.half : 0;
            s0 = sp.interp ? sc : sn;
            ds = sp.dshift;
            h = sp.dZ * HDZ_SCALE;
        }
        // the sub-points lo < m <= hi lie inside the window
        const int lo = span == SPAN_NONE ? n : (int)(((span & 255) * (unsigned)n) >> 8);
        const int hi = span == SPAN_NONE ? 0 : (int)((((span >> 8) + 1) * (unsigned)n + 255) >> 8);
        // the interval before an inward step's first point, or the origin, is the previous step's
        double h_in = from_lane(h, lane - 1);
        if (lane == 0) h_in = h_last;
        if (outward) h_in = h;
        h_last = from_lane(h, WAVE - 1);
        const int incl = scan_add(n), base = incl - n;
        int total = __builtin_amdgcn_readlane(incl, WAVE - 1);
        total = total < left ? total : left;
        left -= total;
        for (int w0 = 0; w0 < total; w0 += W) {
            const int cw = total - w0 < W ? total - w0 : W;
            wave_lds_fence();   // the previous window is consumed
            win.owner[lane] = 0;
            wave_lds_fence();
            // (base, lane) of the step that begins at a point, or before the window and ends in it
            if (n > 0 && base < w0 + W && base + n > w0) win.owner[base > w0 ? base - w0 : 0] = base << 6 | lane;
            wave_lds_fence();
            const int bl = scan_max(win.owner[lane]);
            const int own = bl & (WAVE - 1);
            const int k = w0 + lane - (bl >> 6);   // the point's number in its step, in visiting order
            const int o_n = from_lane(n, own);
            const int m = g0 + own < nsx ? o_n - k : k + 1;
            Stage<double> sg;
            sg.s = sub_point_shift(from_lane(s0, own), m, from_lane(ds, own));
            const int32_t c_own = from_lane(c_next, own), c_before = from_lane(c_prev, own);
            sg.cell = m < from_lane(half, own) ? c_before : c_own;
            const int o_lo = from_lane(lo, own), o_hi = from_lane(hi, own);   // on every lane, before the || below
            const uint64_t floors = __ballot(m <= o_lo || m > o_hi);
            const double h_own = from_lane(h, own), h_first = from_lane(h_in, own);
            win.hdz[lane] = k == 0 ? h_first : h_own;
            win.stage[lane] = sg;
            wave_lds_fence();
            {
                // the rows of WAVE / L points at a time, lane e L + l line l of point e
                const int per = WAVE / L;
                const int e0 = (int)(((uint64_t)(uint32_t)lane * ka->L_magic) >> 32), l = lane - e0 * L;
                const double4 *src = ka->rows + l;
                double4 *dst = win.rows + l * (W + 1);
                if (e0 < per)
                    for (int e = e0; e < cw; e += per) {
                        if ((floors >> e) & 1) continue;
                        const Stage<double> sg_e = win.stage[e];
                        const double4 v = src[(uint32_t)sg_e.cell * (uint32_t)L];   // N L rows < 2^32
                        dst[e] = make_double4(ONE ? sg_e.s : v.x, v.y, v.z, v.w);
                    }
            }
            wave_lds_fence();
            for (int p = 0; p < cw; ++p) {
                double eta = 0.0, chi = CHI_FLOOR * CHI_SCALE;
                if (!((floors >> p) & 1)) eval_window<double, ONE>(a, lc, win, p, W, eta, chi);
                visit(t++, eta, chi, win.hdz[p], p);
            }
        }
    }
}

// Image of ray r (Simulation::compute_and_write_image, sim_radiation.tpp:345-478;
// RayPair::solve_for_image, raypair_solver.tpp:523-579).  Entries 2o (the
// antipode, index 0 end of the pair) and 2o + 1 (ray r, index ndep-1 end) of
// the rest-frame trace.  The intensities leaving the pair are
// I_p = 2 u(ndep-1) - I_bdy_n and I_m = 2 u(0) - I_bdy_0 (RayPair::get_Ip_at_end,
// get_Im_at_front, raypair.tpp:212-229).
// u at the end of the elimination is its boundary row's.  The rows say
// u_n = q_n u_{n+1} + c_n z_n, so u_0 = U + P u_n with P the product of the q
// and U the sum of P c z: one sweep for both ends, no per-point storage.
//
// FP64: one wave per (origin, chunk of bins), at 4 per SIMD.  Bound by the
// evaluation of every point, most of them outside the window of most bins.  Two
// sweeps by workgroups that staged 64 steps at a time (as k_image32) took 5.2 ms
// at 36^3 cells and 186 bins, this takes 2.3.
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_image64(RFArgs<double> a,
                                                                                          double *__restrict__ I_m,
                                                                                          double *__restrict__ I_p)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int G = gridDim.x;
    const int per = G >> 3;
    const int bid = blockIdx.x;
    const int logical = (bid & 7) * per + (bid >> 3);
    if (logical >= a.grid_real) return;
    const int32_t o = a.o_begin + (int32_t)(logical / a.nchunk);
    const int chunk = logical - (o - a.o_begin) * a.nchunk;
    const int lane = (int)threadIdx.x;
    Window<double> win;
    win.place(smem);
    const int F = a.F;
    const int f = chunk * WAVE + lane;
    const bool active = f < F;
    const int fa = active ? f : F - 1;
    const double nu_f = a.nu[(int64_t)o * F + fa];
    const double dsm = a.dshift_max[o];
    const int32_t bo = a.cell2bdy[o];
    LaneCtx<double> lc;
    {
        // the line frequencies, read at every point
        double *lt = reinterpret_cast<double *>(smem + a.line_offset);
        for (int i = lane; i < a.L; i += WAVE) lt[i] = a.tb->line[i];
        wave_lds_fence();
        lc.line = lt;
    }
    double S_o, chi_o;
    origin_point<double>(a, nu_f, a.rows + (int64_t)o * a.L, lc, S_o, chi_o);

    int32_t err = 0;
    const int64_t qa = 2 * (int64_t)o, qr = qa + 1;
    const int n_a = rfl_int(a.npts[qa]);
    const int n_r = rfl_int(a.npts[qr]);
    double Im = 0.0, Ip = 0.0;
    if (n_a == 0 && n_r == 0) {
        // too short a ray: both intensities are I_bdy of the origin's boundary entry
        if (bo < 0) err |= ERR_EMPTY_SIDE;
        else Im = Ip = a.I_bdy[(int64_t)bo * F + fa];
    } else {
        double I_o = 0.0;   // an empty side takes I_bdy of the origin's boundary entry
        if (n_a == 0 || n_r == 0) {
            if (bo < 0) err |= ERR_EMPTY_SIDE;
            else I_o = a.I_bdy[(int64_t)bo * F + fa];
        }
        const double I0 = n_a > 0 ? far_intensity(a, qa, nu_f, F, err) : I_o;
        const double In = n_r > 0 ? far_intensity(a, qr, nu_f, F, err) : I_o;
        Sweep<double> sw;
        sw.init(I0 * I_SCALE);
        double U = 0.0, P = 1.0;
        walk_pair<false>(a, lc, o, qa, qr, n_r, dsm, chunk, win, [&](int t, double eta, double chi, double h, int) {
            const double S = eta * Prec<double>::rcp(chi);
            if (t <= n_a) {   // inwards and to the origin, with the pending point's path factor
                sw.hdz_q = h;
                sw.cq = sw.chi_q * h;
                sw.step(chi);
            } else {
                sw.step_out(chi, h);
            }
            sw.pend(S, chi, h);
            U = fmad(P, sw.c * sw.z, U);
            P *= sw.q;
        });
        const double u_n = end_u(sw, In * I_SCALE), u_0 = fmad(P, u_n, U);
        Ip = 2.0 * (u_n * (1.0 / I_SCALE)) - In;
        Im = 2.0 * (u_0 * (1.0 / I_SCALE)) - I0;
    }
    if (err) atomicOr(a.err_flag, err);
    if (active) {
        I_m[(int64_t)o * F + f] = Im;
        I_p[(int64_t)o * F + f] = Ip;
    }
}

// The same in FP32, with shifts and profile arguments in FP64 (eta_chi32x).
// Instead of a stored forward elimination and back-substitution, each end's u
// comes from one full sweep that starts at the other end, passes the origin and
// closes at the end itself with its boundary row: two sweeps, no per-point
// storage.  (36^3 cells, 186 bins: 1.18 ms; on walk_pair 1.35.)
__global__ __launch_bounds__(WAVE * MAX_WAVES) void k_image32(RFArgs<float> a, double *__restrict__ I_m,
                                                              double *__restrict__ I_p)
{
    extern __shared__ __align__(16) unsigned char smem[];
    Step *st = reinterpret_cast<Step *>(smem);
    float4 *rw = reinterpret_cast<float4 *>(smem + a.row_offset);

    const int G = gridDim.x;
    const int per = G >> 3;
    const int bid = blockIdx.x;
    const int logical = (bid & 7) * per + (bid >> 3);
    if (logical >= a.grid_real) return;   // whole workgroup: before any barrier
    const int32_t o = a.o_begin + (int32_t)(logical / a.ngroups);
    const int group = logical - (o - a.o_begin) * a.ngroups;
    const int wave = threadIdx.x / WAVE;
    const int chunk = rfl_int(group * a.nwg + wave);   // wave-uniform: scalar skip tests
    const int F = a.F;
    const int f = chunk * WAVE + (int)(threadIdx.x & (WAVE - 1));
    const bool active = f < F;
    const int fa = active ? f : F - 1;
    const double nu_f = a.nu[(int64_t)o * F + fa];
    const double dsm = a.dshift_max[o];
    const int32_t bo = a.cell2bdy[o];
    const float4 *orow = a.rows + (int64_t)o * a.L;

    LaneCtx<float> lc;
    float S_o, chi_o;
    origin_point<float, true>(a, nu_f, orow, lc, S_o, chi_o);

    int32_t err = 0;
    const int64_t qa = 2 * (int64_t)o, qr = qa + 1;
    const int n_a = a.npts[qa];
    const int n_r = a.npts[qr];
    double Im = 0.0, Ip = 0.0;
    if (n_a == 0 && n_r == 0) {
        // too short a ray: both intensities are I_bdy of the origin's boundary entry
        if (bo < 0) err |= ERR_EMPTY_SIDE;
        else Im = Ip = a.I_bdy[(int64_t)bo * F + fa];
    } else {
        double I_o = 0.0;   // an empty side takes I_bdy of the origin's boundary entry
        if (n_a == 0 || n_r == 0) {
            if (bo < 0) err |= ERR_EMPTY_SIDE;
            else I_o = a.I_bdy[(int64_t)bo * F + fa];
        }
        const double I0 = n_a > 0 ? far_intensity(a, qa, nu_f, F, err) : I_o;
        const double In = n_r > 0 ? far_intensity(a, qr, nu_f, F, err) : I_o;
        const float I0s = (float)(I0 * I_SCALE);
        const float Ins = (float)(In * I_SCALE);
        float u_n, u_0;
        {
            // from the antipode's far end through the origin to ray r's end
            Sweep<float> A;
            if (n_a > 0) {
                A = sweep_side(a, lc, o, qa, I0s, S_o, chi_o, dsm, st, rw);
            } else {
                A.init(I0s);
                A.pend(S_o, chi_o, (float)0);
            }
            sweep_outward(a, lc, o, qr, dsm, A, st, rw);
            u_n = end_u(A, Ins);
        }
        {
            // and back
            Sweep<float> B;
            if (n_r > 0) {
                B = sweep_side(a, lc, o, qr, Ins, S_o, chi_o, dsm, st, rw);
            } else {
                B.init(Ins);
                B.pend(S_o, chi_o, (float)0);
            }
            sweep_outward(a, lc, o, qa, dsm, B, st, rw);
            u_0 = end_u(B, I0s);
        }
        Ip = 2.0 * ((double)u_n * (1.0 / I_SCALE)) - In;
        Im = 2.0 * ((double)u_0 * (1.0 / I_SCALE)) - I0;
    }
    if (err) atomicOr(a.err_flag, err);
    if (active) {
        I_m[(int64_t)o * F + f] = Im;
        I_p[(int64_t)o * F + f] = Ip;
    }
}

// ---- banded Lambda* (n_off_diag >= 2) ------------------------------------------

// The elimination's coefficients along one direction of a pair: close() takes
// the next point and closes the row of the one before it.  With dt the closed
// row's interval and dt' the one before it, c = dt / sqrt 2 and
// F = 0.5 dt (dt + dt') (1 + F' / (0.5 dt' (dt + dt') (1 + F'))), the
// reference's F (or G), is c x: the part of the sweeps' recurrence that no
// source enters, without the divisions by the intervals.  The virtual start
// gives F = dt + dt^2 / 2, the boundary row's.
struct RowSweep {
    double chi = 0.0, c = 0.0, c_prev = 0.0, y = SQRT2;
    double F = 0.0, q = 1.0;   // of the closed row, q = 1 / (1 + F)

    __device__ __forceinline__ void close(double chi_next, double h)
    {
#pragma clang fp contract(off)
        c_prev = c;
        c = (chi + chi_next) * h;
        const double x = c + y;
        F = c * x;
        q = Prec<double>::rcp(1.0 + F);
        y = __builtin_fma(x, q, c);
        chi = chi_next;
    }
    // 1/A or 1/C of the closed row: 0.5 (dt + dt') dt
    __device__ __forceinline__ double inverse_C() const { return (c_prev + c) * c; }
};

// Thermodynamics::profile (thermodynamics.tpp:16-29) of width `width` at
// freq_diff.
__device__ __forceinline__ double profile64(double width, double freq_diff)
{
#pragma clang fp contract(off)
    const double iw = Prec<double>::rcp(width);
    const double x = iw * freq_diff;
    return iw * INVERSE_SQRT_PI * exp_neg(x * x);
}

// The band elements of Lambda* (RayPair::update_Lambda, raypair_lambda.tpp:129-146,
// with get_L_lower / get_L_upper, raypair_lambda.tpp:44-84) in FP64.  One wave
// of 64 bins per (origin, chunk of bins).  Per ray pair the longer ray is the
// low side (n_ar = nA points, sim_radiation.tpp:164-171), and for band
// m = 1 .. nband
//   lower: L_lower[m][n_ar-m] = L_diag[n_ar-m] prod_{q=n_ar-m+1}^{n_ar+1} 1/(1+G_q),
//   upper: L_upper[m][n_ar+m] = L_diag[n_ar+2m+1] prod_{q=n_ar+2m}^{n_ar+m} 1/(1+F_q),
//   L_diag[n] = 1/C_n / (F_n + G_{n+1} / (1 + G_{n+1})),
// each times A_k (w_z 2 w_r) nu phi(nu) / chi at its own point, where the
// pair's solve wrote it (the slots k_band_cells marks).
//   pass 1, from index last down to n_ar - nband: G, of which the products and
//   the terms of L_diag that the elements need go to LDS;
//   pass 2, from index 0 up to n_ar + 2 nband + 2: F and the elements.
// Both passes walk the pair as the field kernel does (walk_pair), and the
// lanes' elements are added per transition from LDS, one lane per (element,
// transition); k_band_sum adds the waves of an origin.
//
// Bound by the FP64 profile and recurrence of every point, at 4 waves per SIMD
// (125 VGPRs, 8 KB of LDS).  A walk with per-step scalar loads and divisions in
// every lane, three rcp per point, five arrays of 3 (nband + 1) points in LDS
// and butterfly sums per element and transition took 9.5 ms at 20^3 cells, 84
// bins and one band; this one takes 3.4 ms.
template <bool ONE>
__global__ __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(4))) void k_lambda_band(RFArgs<double> a)
{
#pragma clang fp contract(off)
    extern __shared__ __align__(16) unsigned char smem[];
    const int G = gridDim.x;
    const int per = G >> 3;
    const int bid = blockIdx.x;
    const int logical = (bid & 7) * per + (bid >> 3);
    if (logical >= a.grid_real) return;
    const int32_t o = (int32_t)(logical / a.nchunk);
    const int chunk = logical - o * a.nchunk;
    const int lane = (int)threadIdx.x;
    const int F = a.F, L = a.L, nb = a.nband;
    Window<double> win;
    win.place(smem);
    // per band and lane: elem [2 nb] the elements, lower ones first (before them
    // the products over G or F so far), termG [2 nb] G / (1 + G) for their L_diag
    double *elem = reinterpret_cast<double *>(win.rows + (size_t)L * (a.ch + 1));
    double *termG = elem + 2 * nb * WAVE;
    double *lt = termG + 2 * nb * WAVE;   // the line frequencies
    int *first = reinterpret_cast<int *>(lt + L);   // [L + 1] of the transitions in elem's order of summation
    // the lane order of the field kernels (lane_bin), which the out-of-window bits follow
    const int slot = chunk * WAVE + lane;
    const bool active = slot < F;
    const int fa = lane_bin(active ? slot : F - 1, L, F, a.root_major);
    const int k = active ? a.f_k[fa] : L;
    const double nu_f = a.nu[(int64_t)o * F + fa];
    const double dsm = a.dshift_max[o];
    LaneCtx<double> lc;
    for (int i = lane; i < L; i += WAVE) lt[i] = a.tb->line[i];
    lc.line = lt;
    // lanes in order of their transition
    int pos = 0, sorted = 0;
    for (int kk = 0; kk <= L; kk++) {
        const uint64_t same = __ballot(k == kk);
        if (k == kk) pos = sorted + __builtin_popcountll(same & ((1ull << lane) - 1));
        if (lane == 0) first[kk] = sorted;
        sorted += __builtin_popcountll(same);
    }
    wave_lds_fence();
    double S_o, chi_o;
    origin_point<double, false, ONE>(a, nu_f, a.rows + (int64_t)o * L, lc, S_o, chi_o);
    const double freq_line = k < L ? a.freq_k[k] : nu_f;
    const double A_k = k < L ? a.A_k[k] : 0.0;
    const double w_z = k < L ? a.qw[a.f_z[fa]] : 0.0;
    const int64_t qb = a.cell_qbase[o];
    const int Rh = a.m_R[0] / 2;
    double *part = a.band_part + ((int64_t)o * a.nchunk + chunk) * a.band_S * L;

    for (int r = 0; r < Rh; r++) {
        const int64_t qr = qb + r, qa = qb + a.antipod[r];
        const int n_r = rfl_int(a.npts[qr]), n_a = rfl_int(a.npts[qa]);
        const bool r_longer = n_r > n_a;
        const int64_t qA = r_longer ? qr : qa, qB = r_longer ? qa : qr;
        const int nA = r_longer ? n_r : n_a, nB = r_longer ? n_a : n_r;
        const int last = nA + nB;
        const double factor = A_k * (w_z * 2.0 * a.ray_w[r]);
        wave_lds_fence();   // the last pair's elements are summed
        if (nB >= 1) {
            RowSweep sw;
            double prod = 1.0;
            walk_pair<ONE>(a, lc, o, qB, qA, nA < nb ? nA : nb, dsm, chunk, win,
                           [&](int t, double, double chi, double h, int) {
                sw.close(chi, h);   // row last - t + 1 (none at t = 0)
                const int i = last - t + 1 - nA;
                if (i > 2 * nb + 2 || t == 0) return;
                if (i >= 4 && !(i & 1)) termG[(nb + i / 2 - 2) * WAVE + lane] = sw.F * sw.q;   // of band i/2 - 1
                if (i <= 1) {
                    prod *= sw.q;
                    if (i <= 0) {   // of band 1 - i
                        elem[-i * WAVE + lane] = prod;
                        termG[-i * WAVE + lane] = sw.F * sw.q;
                    }
                }
            });
            sw = RowSweep();
            double fpc = 0.0;   // nu phi(nu) / chi of the last point, factor applied
            const int ny = nB < 2 * nb + 2 ? nB : 2 * nb + 2;
            walk_pair<ONE>(a, lc, o, qA, qB, ny, dsm, chunk, win, [&](int n, double, double chi, double h, int p) {
                sw.close(chi, h);   // row n - 1 (none at n = 0)
                const int i = n - 1 - nA;
                if (i < -nb - 1) return;
                if (i < 0) {
                    if (i >= -nb && n > 0) {   // lower element of band -i
                        const int at = (-i - 1) * WAVE;
                        const double T = sw.inverse_C() * Prec<double>::rcp(sw.F + termG[at + lane]) * elem[at + lane];
                        elem[at + pos] = fpc * T;
                    }
                } else if (i > 0) {
                    // the products of the bands m with i in m .. 2 m
                    for (int m = (i + 1) / 2; m <= nb && m <= i; m++) {
                        double &e = elem[(nb + m - 1) * WAVE + lane];
                        e = (m == i ? fpc : e) * sw.q;
                    }
                    const int m = i >> 1;
                    if (m >= 1 && m <= nb) {
                        const int at = (nb + m - 1) * WAVE;
                        if (i & 1) {   // upper element of band m, from row n_ar + 2m + 1
                            const double T = sw.inverse_C() * Prec<double>::rcp(sw.F + termG[at + lane]);
                            elem[at + pos] = elem[at + lane] * T;
                        } else if (n == last) {   // which is the last row
                            const double c2 = sw.c * sw.c;
                            const double T = c2 * Prec<double>::rcp(c2 + SQRT2 * sw.c + sw.F * sw.q);
                            elem[at + pos] = elem[at + lane] * T;
                        }
                    }
                }
                // nu phi(nu) / chi at the point's own cell and frequency, where an element needs it
                if (i < -1 || (i >= 0 && i < nb && nB > 2 * (i + 1))) {
                    const Stage<double> sg = win.stage[p];
                    const double fs = sg.s * nu_f;
                    fpc = factor * (fs * profile64(freq_line * a.pw[sg.cell], fs - freq_line)) *
                          Prec<double>::rcp(chi * (1.0 / CHI_SCALE));
                }
            });
        }
        // elements that the pair does not have
        for (int m = 1; m <= nb; m++) {
            if (nB < 1 || nA < m) elem[(m - 1) * WAVE + lane] = 0.0;
            if (nB <= 2 * m) elem[(nb + m - 1) * WAVE + lane] = 0.0;
        }
        wave_lds_fence();
        for (int s = lane; s < 2 * nb * L; s += WAVE) {
            const int i = s / L, kk = s - i * L;
            double sum = 0.0;
            for (int u = first[kk]; u < first[kk + 1]; u++) sum += elem[i * WAVE + u];
            part[(int64_t)r * 2 * nb * L + s] = sum;
        }
    }
}

// Band sums per (origin, slot, transition): the waves of an origin in chunk order.
__global__ void k_band_sum(int64_t N, int64_t SL, int nchunk, const double *__restrict__ part,
                           double *__restrict__ out)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N * SL) return;
    const int64_t o = t / SL, i = t - o * SL;
    double acc = 0.0;
    for (int c = 0; c < nchunk; c++) acc += part[(o * nchunk + c) * SL + i];
    out[t] = acc;
}

// Largest chunk of staged steps that fits the LDS budget with the cells'
// line rows, at most CH_MAX: also the most points that a launch shape can ask for.
template <typename real>
int max_chunk(const mgr_ctx *ctx)
{
    const size_t per_entry = sizeof(Step) + sizeof(typename Prec<real>::row_t) * ctx->L + 64;
    const int ch = (int)(LDS_LIMIT / per_entry) - 1;
    return ch < CH_MAX ? ch : CH_MAX;
}

// A line can be inside the window of bin nu_f at some point only if
// nu_l (1 - 11 pw_max) <= s_max nu_f and nu_l (1 + 11 pw_max) >= s_min nu_f, with
// shifts in [shift_min, shift_max]: line * lo < nu_f is below the bin's reach,
// line * hi <= nu_f a candidate.  The margins cover rounding of the shifts and widths.
void candidate_bounds(const mgr_ctx *ctx, double shift_min, double shift_max, double &lo, double &hi)
{
    const double w = LINE_WINDOW * ctx->pw_max;
    lo = (1.0 + w) * (1.0 + 1.0e-9) / shift_min;
    hi = (1.0 - w) * (1.0 - 1.0e-9) / shift_max;
}

// Arguments shared by the radiation-field and image kernels: model tables,
// rows, candidate-line bounds for shifts in [shift_min, shift_max], launch
// shape (nwg waves of 64 bins per workgroup, chunks of ch staged steps) over
// origins [o_begin, o_begin + o_count).  The trace pointers are the caller's.
template <typename real>
int make_args(mgr_ctx *ctx, const typename Prec<real>::row_t *rows, int nwg, int ch, int64_t o_begin,
              int64_t o_count, double shift_min, double shift_max, RFArgs<real> &a)
{
    a = RFArgs<real>();
    a.N = ctx->N;
    a.cell_model = ctx->d_cell_model;
    a.cell_qbase = ctx->d_cell_qbase;
    a.m_R = ctx->d_m_R;
    a.m_rbase = ctx->d_m_rbase;
    a.m_active = ctx->d_m_active;
    a.F = (int)ctx->F;
    a.L = (int)ctx->L;
    a.L_magic = 0xFFFFFFFFull / (uint64_t)ctx->L + 1;
    a.nchunk = (int)((ctx->F + WAVE - 1) / WAVE);
    a.nwg = nwg;
    a.ngroups = (a.nchunk + a.nwg - 1) / a.nwg;
    a.o_begin = (int32_t)o_begin;
    a.pair_stride = 1;
    a.tb = ctx->tables;
    a.nu = ctx->nu;
    a.rows = rows;
    a.cell2bdy = ctx->cell2bdy;
    a.antipod = ctx->d_antipod;
    a.I_bdy = ctx->I_bdy;
    a.ray_w = ctx->ray_w;
    a.dshift_max = ctx->dshift_max;
    candidate_bounds(ctx, shift_min, shift_max, a.cand_lo, a.cand_hi);
    a.lstart_threshold = a.cand_lo;
    a.J = ctx->J;
    a.Lam = ctx->Lam;
    a.f_k = ctx->f_k;
    a.f_z = ctx->f_z;
    a.qw = ctx->qweights;
    a.A_k = ctx->A;
    a.freq_k = ctx->frequency;
    a.pw = ctx->pw;
    a.Lpart = ctx->Lpart;
    a.err_flag = ctx->err_flag;
    if (nwg < 1 || nwg > MAX_WAVES || o_begin < 0 || o_count < 1 || o_begin + o_count > ctx->N)
        return ctx->fail(MGR_ERR_ARGUMENT, "radiation-field launch shape out of range");
    const int64_t groups = o_count * a.ngroups;
    if (groups > INT32_MAX - 8) return ctx->fail(MGR_ERR_UNSUPPORTED, "too many workgroups");
    a.grid_real = (int)groups;
    if (ch < 2 || ch > max_chunk<real>(ctx)) return ctx->fail(MGR_ERR_UNSUPPORTED, "line rows do not fit the LDS budget");
    a.ch = ch;
    a.row_offset = ((sizeof(Step) * (ch + 1) + 63) / 64) * 64;
    return MGR_OK;
}

// LDS of the field kernel with nwg waves per workgroup: the window of each wave
// (of up to `points` points), then the line table.
template <typename real>
FieldLds window_lds(const mgr_ctx *ctx, int nwg, int points)
{
    return field_lds(Window<real>::fixed, sizeof(typename Prec<real>::row_t) * ctx->L, sizeof(double) * ctx->L, nwg,
                     points);
}

// One candidate line per bin of the co-moving frame: the lines' candidate ranges
// are disjoint.
bool one_line(const mgr_ctx *ctx)
{
    double lo, hi;
    candidate_bounds(ctx, ctx->shift_min, ctx->shift_max, lo, hi);
    for (int l = 0; l + 1 < ctx->h_tables.L; l++)
        if (!(ctx->h_tables.line[l] * lo <= ctx->h_tables.line[l + 1] * hi)) return false;
    return true;
}

// Points per window of walk_pair: at most 32, with rows of up to 8 KB, so that 4
// waves fit a SIMD.
int walk_window(const mgr_ctx *ctx)
{
    const int64_t row = sizeof(double4) * ctx->L;
    return (int)std::max<int64_t>(2, std::min<int64_t>(32, 8 * 1024 / row - 1));
}

template <typename real>
unsigned grid_of(const RFArgs<real> &a)
{
    return (unsigned)(((int64_t)a.grid_real + 7) / 8) * 8;
}

// The range of y in which the points of an out-of-window run change nothing
// (Runs), with chi at most X times the floor there; empty (lo > hi) if there is
// none.  Such a point closes its row with c = chi dz'_a + chi' dz'_b (rounded
// twice), at most cb = 2 X dz'_max (1 + 2^-20).  The no-op needs cb < y 2^-25
// (then c is below half an ulp of y) and cb y < 2^-25 (then 1 + c y rounds to 1).
void noop_range(const mgr_ctx *ctx, double X, float &lo_out, float &hi_out)
{
    lo_out = INFINITY;   // never
    hi_out = 0.0f;
    if (!(ctx->hdz32_max > 0.0f)) return;
    const double cb = 2.0 * X * (double)(float)(CHI_FLOOR * CHI_SCALE) * (double)ctx->hdz32_max * (1.0 + 0x1p-20);
    const double lo = cb * 0x1p25 * (1.0 + 0x1p-20), hi = 0x1p-25 / cb * (1.0 - 0x1p-20);
    if (lo < hi && lo < 3.0e38 && hi > 1.0e-37) {
        lo_out = std::nextafter((float)lo, INFINITY);   // float(lo) may round below lo
        hi_out = std::nextafter((float)hi, 0.0f);
    }
}

// FP32: whether the points are laid out per lane (k_radiation_field) or the steps
// staged for the workgroup (k_field_staged).  By points a wave brings the rows of
// all lines to LDS for every point that it evaluates, by steps the workgroup does
// once per step.  By points is the faster way where most points are passed over
// and the rows are few, steps staged
//   - where runs cannot be passed over by their spans: behind a dark boundary (36^3
//     envelope at 0.05 K 6.8 ms, by points 7.1), with steps beyond 1e18 m (24^3
//     envelope 2.06, 2.82), and with the skip off (16^3 stress 2.26, 2.65);
//   - from 15 lines on (24^3 envelope, 31 lines 1.11 ms, by points 1.88; 15 lines
//     0.55, 0.59; 14 and 13 lines 0.55, 0.55 and 0.55, 0.54);
//   - with more than 16 chunks of bins, of which five are passed over at all (7 lines,
//     22 chunks 1.49 ms, by points 1.55; 17 chunks 1.15, 1.17; 11 chunks 0.78, 0.76),
//     or with more than those five and 12 lines (6 chunks 0.59, 0.63) or bins of
//     several lines (8 chunks 0.76, 0.91).
bool per_point(const mgr_ctx *ctx)
{
    if (!ctx->masks_valid || !ctx->rf_window_skip || !ctx->rf_spans || !ctx->near_on || ctx->bdy_dark) return false;
    const int64_t nchunk = (ctx->F + WAVE - 1) / WAVE;
    if (ctx->L >= 15 || nchunk > 16) return false;
    if (nchunk > STEP_MASK_CHUNKS && (ctx->L >= 12 || !one_line(ctx))) return false;
    float lo, hi;
    noop_range(ctx, NEAR_X, lo, hi);
    return lo < hi;
}

// The launch shape's place in the context: of the FP32 kernel by points, the FP64
// kernel or the FP32 kernel of staged steps.
int shape_of(const mgr_ctx *ctx, int precision) { return precision == MGR_FP64 ? 1 : per_point(ctx) ? 0 : 2; }

// Launch over origins [o_begin, o_begin + o_count) with nwg waves (64 bins
// each) per workgroup and windows of ch points, or chunks of ch staged steps.
template <typename real>
int launch_rf(mgr_ctx *ctx, const typename Prec<real>::row_t *rows, int nwg, int ch, int64_t o_begin,
              int64_t o_count)
{
    RFArgs<real> a;
    int rc = make_args<real>(ctx, rows, nwg, ch, o_begin, o_count, ctx->shift_min, ctx->shift_max, a);
    if (rc) return rc;
    a.seg_off = ctx->seg_off;
    a.nseg = ctx->nseg;
    a.npts = ctx->npts;
    a.seg_cell = ctx->seg_cell;
    a.seg_shift = ctx->seg_shift;
    a.seg_dZ = ctx->seg_dZ;
    a.seg_f32 = ctx->seg_f32;
    a.seg_hdz32 = ctx->seg_hdz32;
    a.far_cell = ctx->far_cell;
    a.far_shift = ctx->far_shift;
    a.origin_shift = nullptr;
    a.pair_stride = ctx->rf_pair_stride;
    a.u_out = ctx->u_store;
    // the out-of-window bits of the kernel's precision (each exact for its own profile)
    if constexpr (sizeof(real) == 4)
        a.step_mask = (ctx->masks_valid && ctx->rf_window_skip) ? ctx->step_mask : nullptr;
    else
        a.step_mask = (ctx->masks64_valid && ctx->rf_window_skip) ? ctx->step_mask64 : nullptr;
    bool by_point = true;
    if constexpr (sizeof(real) == 4) {
        by_point = per_point(ctx);
        noop_range(ctx, by_point ? NEAR_X : 1.0, a.noop_lo, a.noop_hi);
    }
    a.span_stride = ctx->span_stride;
    if (sizeof(real) == 8 && a.step_mask && ctx->rf_spans) a.span = ctx->span64;
    if (sizeof(real) == 4 && by_point) {
        a.span = ctx->span32;
        a.near_p = ctx->near_p;
        a.near_bad = ctx->near_bad;
    }
    a.root_major = ctx->root_major;
    a.far32 = (sizeof(real) == 4 && ctx->far_cache && ctx->far_valid[0]) ? ctx->far_I32 : nullptr;
    a.far64 = (sizeof(real) == 8 && ctx->far_cache && ctx->far_valid[1]) ? ctx->far_I64 : nullptr;
    const bool one = one_line(ctx);
    if constexpr (sizeof(real) == 4) {
        if (!by_point) {
            a.line_offset = a.row_offset + sizeof(float4) * (a.ch + 1) * ctx->L;
            const size_t lds = a.line_offset + (one ? 0 : sizeof(double) * ctx->L);
            auto kernel = one ? k_field_staged<true> : k_field_staged<false>;
            hipLaunchKernelGGL(kernel, dim3(grid_of(a)), dim3(WAVE * a.nwg), lds, ctx->stream, a);
            ctx->last_rf_kernel = one ? "k_field_staged<true>" : "k_field_staged<false>";
            MGR_LAUNCH_CHECK();
            return MGR_OK;
        }
    }
    const FieldLds lds = window_lds<real>(ctx, a.nwg, a.ch);
    if (lds.points < 2) return ctx->fail(MGR_ERR_UNSUPPORTED, "line rows do not fit the LDS budget");
    a.ch = lds.points;
    a.wave_lds = (int)lds.wave;
    a.line_offset = lds.wave * a.nwg;
    auto kernel = one ? k_radiation_field<real, true> : k_radiation_field<real, false>;
    hipLaunchKernelGGL(kernel, dim3(grid_of(a)), dim3(WAVE * a.nwg), lds.total, ctx->stream, a);
    ctx->last_rf_kernel = sizeof(real) == 4 ? (one ? "k_radiation_field<float, true>" : "k_radiation_field<float, false>")
                                            : (one ? "k_radiation_field<double, true>" : "k_radiation_field<double, false>");
    MGR_LAUNCH_CHECK();
    return MGR_OK;
}

// Image kernel over every origin, on the rest-frame trace of ctx->img.  FP32: the
// sweep and profiles in FP32, shifts and profile arguments in FP64.
template <typename real>
int launch_image(mgr_ctx *ctx, const typename Prec<real>::row_t *rows)
{
    constexpr bool F32 = sizeof(real) == 4;
    const int nchunk = (int)((ctx->F + WAVE - 1) / WAVE);
    const mgr_ctx::ImageTrace &g = ctx->img;
    RFArgs<real> a;
    int rc = make_args<real>(ctx, rows, F32 ? std::min(nchunk, MAX_WAVES) : 1, max_chunk<real>(ctx), 0,
                                  ctx->N, g.shift_min, g.shift_max, a);
    if (rc) return rc;
    a.step_mask = nullptr;   // the masks index the co-moving cache, not the image's trace
    a.seg_off = g.seg_off;
    a.nseg = g.nseg;
    a.npts = g.npts;
    a.seg_cell = g.seg_cell;
    a.seg_shift = g.seg_shift;
    a.seg_dZ = g.seg_dZ;
    a.far_cell = g.far_cell;
    a.far_shift = g.far_shift;
    a.origin_shift = g.origin_shift;
    if constexpr (F32) {
        const size_t lds = a.row_offset + sizeof(float4) * (a.ch + 1) * ctx->L;
        hipLaunchKernelGGL(k_image32, dim3(grid_of(a)), dim3(WAVE * a.nwg), lds, ctx->stream, a, g.I_m, g.I_p);
    } else {
        a.ch = walk_window(ctx);
        a.line_offset = Window<double>::bytes(ctx->L, a.ch);
        const size_t lds = a.line_offset + sizeof(double) * ctx->L;
        hipLaunchKernelGGL(k_image64, dim3(grid_of(a)), dim3(WAVE), lds, ctx->stream, a, g.I_m, g.I_p);
    }
    MGR_LAUNCH_CHECK();
    return MGR_OK;
}

}  // namespace

namespace mgr {

// Band elements of Lambda* for the current populations (n_off_diag >= 2):
// k_lambda_band into per-wave shares, then their sums per slot and transition.
int launch_band(mgr_ctx *ctx)
{
    if (ctx->nband <= 0) return MGR_OK;
    RFArgs<double> a;
    int rc = make_args<double>(ctx, ctx->row64, 1, 2, 0, ctx->N, ctx->shift_min, ctx->shift_max, a);
    if (rc) return rc;
    a.seg_off = ctx->seg_off;
    a.nseg = ctx->nseg;
    a.npts = ctx->npts;
    a.seg_cell = ctx->seg_cell;
    a.seg_shift = ctx->seg_shift;
    a.seg_dZ = ctx->seg_dZ;
    a.nband = ctx->nband;
    a.band_S = ctx->band_S;
    a.band_part = ctx->band_part;
    a.root_major = ctx->root_major;
    a.span_stride = ctx->span_stride;
    if (ctx->masks64_valid && ctx->rf_window_skip) {
        a.step_mask = ctx->step_mask64;
        if (ctx->rf_spans) a.span = ctx->span64;
    }
    a.ch = walk_window(ctx);
    const size_t lds = Window<double>::bytes(ctx->L, a.ch) +
                       sizeof(double) * (4 * (size_t)ctx->nband * WAVE + ctx->L) + sizeof(int) * (ctx->L + 1);
    auto kernel = one_line(ctx) ? k_lambda_band<true> : k_lambda_band<false>;
    hipLaunchKernelGGL(kernel, dim3(grid_of(a)), dim3(WAVE), lds, ctx->stream, a);
    MGR_LAUNCH_CHECK();
    const int64_t SL = ctx->band_S * ctx->L;
    hipLaunchKernelGGL(k_band_sum, dim3((unsigned)((ctx->N * SL + 255) / 256)), dim3(256), 0, ctx->stream, ctx->N,
                       SL, a.nchunk, ctx->band_part, ctx->band_Ls);
    MGR_LAUNCH_CHECK();
    return MGR_OK;
}

template <typename real>
static int launch_rf_shape(mgr_ctx *ctx, int nwg, int ch, int64_t o_begin, int64_t o_count)
{
    if constexpr (sizeof(real) == 8)
        return launch_rf<double>(ctx, ctx->row64, nwg, ch, o_begin, o_count);
    else
        return launch_rf<float>(ctx, ctx->row32, nwg, ch, o_begin, o_count);
}

// The largest window whose LDS still admits the waves that the kernel's
// registers do, 8, 6 or 4 per SIMD: a pair's points take the fewest windows
// there.  FP32 at 64^3 cells (6 lines, 41 points): 31.4 ms against 31.9 with 32
// points, and 34.1 with 48, which only 26 waves per CU have room for.  FP64 at
// 24^3 cells with 31 lines (7 points): 3.75 ms with 6 points, 5.2 with 16, and 6.95
// with 7, whose rows lie 8 apart and meet in the same banks.
template <typename real>
static int fitting_window(const mgr_ctx *ctx)
{
    constexpr size_t CU_LDS = 160 * 1024, GRANULE = 1280;
    const size_t waves = 4 * (sizeof(real) == 8 ? 4 : one_line(ctx) ? 8 : 6);
    const size_t room = CU_LDS / waves / GRANULE * GRANULE, table = sizeof(double) * ctx->L;
    const size_t row = sizeof(typename Prec<real>::row_t) * ctx->L;
    // a wave's LDS is rounded up to 64 bytes
    if (room < Window<real>::fixed + table + 64 + 3 * row) return 2;
    return (int)std::min<size_t>(64, (room - table - Window<real>::fixed) / 64 * 64 / row - 1);
}

// Launch-shape autotuner: points per window first, with one wave (a 64-bin
// chunk) per workgroup, then waves per workgroup with the best window.  Timed
// on two slices of origins, around 1/8 and 5/8 of the model's cells, so that
// outer and inner cells are seen, each with the waves the chip holds at once;
// smaller models are timed whole.  The fastest shape (or the one with the
// fewest waves among near-ties) is kept for the context and precision.  Runs
// outside graph capture, before the first radiation field of a precision.
//
// What is tried is what has won somewhere: 64-point windows only where the
// waves do not fill the chip twice (56 against 59 us at 10^3 cells; 10 to 25 %
// behind on every larger model), and several waves per workgroup, which share
// only the line table, only where bins meet several lines (6 % ahead on the
// blended model; with one line equal or up to 12 % behind).  A 27^3-cell solve
// takes 24 to 25 ms with these 2 shapes, 27 with 4, and 48 with all combinations
// on 16384 origins and the best ones again on the whole model.
template <typename real>
static int tune(mgr_ctx *ctx, int pi)
{
    const bool staged = pi == 2;
    const int nchunk = (int)((ctx->F + WAVE - 1) / WAVE);
    const int chmax = max_chunk<real>(ctx);
    if (chmax < 2) return ctx->fail(MGR_ERR_UNSUPPORTED, "line rows do not fit the LDS budget");
    const int64_t fill = (WAVES_IN_FLIGHT + nchunk - 1) / nchunk;   // origins that fill the chip
    const int nslice = ctx->N > 2 * fill ? 2 : 1;
    const int64_t per = nslice == 2 ? fill : ctx->N;
    const int fit = std::min(fitting_window<real>(ctx), chmax);
    std::vector<int> chs{std::min(16, chmax)}, nwgs;
    if (staged) {
        if (chmax > 16) chs.push_back(std::min(32, chmax));
        if (chmax > 32) chs.push_back(chmax);
    } else {
        // smaller with many lines, then even: the lines' rows are points + 1 apart
        if (fit > chs.front()) chs.push_back(fit);
        else if (fit < chs.front()) chs.push_back(std::max(fit / 2 * 2, 2));
        if (nslice == 1 && chmax > std::max(fit, chs.front())) chs.push_back(chmax);
    }
    if (staged || !one_line(ctx))
        for (int w = 2; w <= MAX_WAVES; w++)
            if (w == nchunk || (nchunk % w) == 0 || w == std::min(nchunk, MAX_WAVES)) nwgs.push_back(w);
    auto launch_slices = [&](int w, int c) {
        if (nslice == 1) return launch_rf_shape<real>(ctx, w, c, 0, ctx->N);
        int r = launch_rf_shape<real>(ctx, w, c, std::max<int64_t>(ctx->N / 8 - per / 2, 0), per);
        if (!r) r = launch_rf_shape<real>(ctx, w, c, std::min(ctx->N * 5 / 8 - per / 2, ctx->N - per), per);
        return r;
    };
    hipEvent_t e0, e1;
    MGR_HIP(hipEventCreate(&e0));
    MGR_HIP(hipEventCreate(&e1));
    int best_w = 1, best_c = chs.front();
    float best = 1e30f;
    int rc = launch_slices(1, chs.back());   // warm-up
    ctx->tune_log.clear();
    auto time_shape = [&](int w, int points) {
        const int c = staged ? points : window_lds<real>(ctx, w, points).points;
        if (c < 2) return ctx->fail(MGR_ERR_UNSUPPORTED, "line rows do not fit the LDS budget");
        float ms = 0.0f;
        if (hipEventRecord(e0, ctx->stream) != hipSuccess) return MGR_ERR_DEVICE;
        const int r = launch_slices(w, c);
        if (r) return r;
        if (hipEventRecord(e1, ctx->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
            hipEventElapsedTime(&ms, e0, e1) != hipSuccess)
            return MGR_ERR_DEVICE;
        ctx->tune_log.push_back({w, c, ms});
        // more waves only for 2 % (fewer schedule the end of a full launch more evenly), and more staged steps
        if (ms < best * (w > best_w || (staged && c > best_c) ? 0.98f : 1.0f)) {
            best = ms;
            best_w = w;
            best_c = c;
        }
        return MGR_OK;
    };
    for (size_t i = 0; i < chs.size() && !rc; i++) rc = time_shape(1, chs[i]);
    const int window = best_c;
    for (size_t i = 0; i < nwgs.size() && !rc; i++) {
        if (!staged) rc = time_shape(nwgs[i], window);
        else   // the waves share the steps: every size
            for (size_t k = 0; k < chs.size() && !rc; k++) rc = time_shape(nwgs[i], chs[k]);
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc == MGR_ERR_DEVICE ? ctx->fail(MGR_ERR_DEVICE, "radiation-field tuning failed") : rc;
    ctx->rf_nwg[pi] = best_w;
    ctx->rf_ch[pi] = best_c;
    return MGR_OK;
}

int tune_radiation_field(mgr_ctx *ctx, int precision)
{
    const int pi = shape_of(ctx, precision);
    if (ctx->rf_nwg[pi] > 0) return MGR_OK;
    return pi == 1 ? tune<double>(ctx, pi) : tune<float>(ctx, pi);
}

int launch_rf_kernel(mgr_ctx *ctx, int precision)
{
    const int pi = shape_of(ctx, precision);
    if (ctx->rf_nwg[pi] <= 0) return ctx->fail(MGR_ERR_STATE, "radiation-field launch shape not chosen");
    return pi == 1 ? launch_rf_shape<double>(ctx, ctx->rf_nwg[pi], ctx->rf_ch[pi], 0, ctx->N)
                   : launch_rf_shape<float>(ctx, ctx->rf_nwg[pi], ctx->rf_ch[pi], 0, ctx->N);
}

}  // namespace mgr

extern "C" int mgr_compute_radiation_field(mgr_ctx *ctx, int precision)
{
    if (!ctx) return MGR_ERR_ARGUMENT;
    if (precision != MGR_FP32 && precision != MGR_FP64) return ctx->fail(MGR_ERR_ARGUMENT, "precision must be MGR_FP32 or MGR_FP64");
    if (!ctx->spectral_set) return ctx->fail(MGR_ERR_STATE, "compute_spectral_discretisation first");
    if (!ctx->bdy_set) return ctx->fail(MGR_ERR_STATE, "compute_boundary_intensities first");
    if (!ctx->pops_set) return ctx->fail(MGR_ERR_STATE, "level populations not set");
    MGR_HIP(hipSetDevice(ctx->device));
    if (!ctx->traced) {
        int rc = launch_trace(ctx);
        if (rc) return rc;
    }
    int rc0 = set_active(ctx, true);
    if (!rc0) rc0 = launch_step_masks(ctx, precision == MGR_FP64);
    if (!rc0 && ctx->nband > 0) rc0 = launch_step_masks(ctx, true);   // the band kernel's
    if (!rc0) rc0 = launch_far_cache(ctx, precision);
    if (!rc0) rc0 = tune_radiation_field(ctx, precision);
    if (rc0) return rc0;
    hipEvent_t e0, e1;
    MGR_HIP(hipEventCreate(&e0));
    MGR_HIP(hipEventCreate(&e1));
    MGR_HIP(hipMemsetAsync(ctx->err_flag, 0, sizeof(int32_t), ctx->stream));
    // the events bracket the radiation-field kernel alone
    MGR_HIP(hipEventRecord(e0, ctx->stream));
    int rc = launch_rf_kernel(ctx, precision);
    if (!rc) {
        MGR_HIP(hipEventRecord(e1, ctx->stream));
        rc = launch_band(ctx);
        if (!rc) rc = launch_lambda(ctx);
    }
    if (rc) { (void)hipEventDestroy(e0); (void)hipEventDestroy(e1); return rc; }
    MGR_HIP(hipEventSynchronize(e1));
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    ctx->last_rf_ms = ms;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    MGR_HIP(hipStreamSynchronize(ctx->stream));   // the band elements and Lambda* sums too
    int32_t errv = 0;
    MGR_HIP(hipMemcpy(&errv, ctx->err_flag, sizeof(int32_t), hipMemcpyDeviceToHost));
    if (errv) return ctx->fail(MGR_ERR_TRACE, "a ray pair ended off the boundary or an interior origin has an empty ray");
    ctx->J_set = true;
    return MGR_OK;
}

// The warm start's first pass: a radiation field over every pair_stride-th
// ray pair of each origin (weights scaled by pair_stride) and J_eff.
extern "C" int mgr_first_pass(mgr_ctx *ctx, int precision, int pair_stride)
{
    if (!ctx) return MGR_ERR_ARGUMENT;
    if (precision != MGR_FP32 && precision != MGR_FP64) return ctx->fail(MGR_ERR_ARGUMENT, "precision must be MGR_FP32 or MGR_FP64");
    if (pair_stride < 1) return ctx->fail(MGR_ERR_ARGUMENT, "pair_stride must be at least 1");
    if (!ctx->spectral_set) return ctx->fail(MGR_ERR_STATE, "compute_spectral_discretisation first");
    if (!ctx->bdy_set) return ctx->fail(MGR_ERR_STATE, "compute_boundary_intensities first");
    if (!ctx->pops_set) return ctx->fail(MGR_ERR_STATE, "level populations not set");
    MGR_HIP(hipSetDevice(ctx->device));
    if (!ctx->traced) {
        int rc = launch_trace(ctx);
        if (rc) return rc;
    }
    int rc = set_active(ctx, true);
    if (!rc) rc = launch_step_masks(ctx, precision == MGR_FP64);
    if (!rc && ctx->nband > 0) rc = launch_step_masks(ctx, true);   // the band kernel's
    if (!rc) rc = launch_far_cache(ctx, precision);
    if (!rc) rc = tune_radiation_field(ctx, precision);
    if (rc) return rc;
    MGR_HIP(hipMemsetAsync(ctx->err_flag, 0, sizeof(int32_t), ctx->stream));
    ctx->rf_pair_stride = pair_stride;
    rc = launch_rf_kernel(ctx, precision);
    ctx->rf_pair_stride = 1;
    if (!rc) rc = launch_band(ctx);
    if (!rc) rc = launch_jeff(ctx, true);
    if (rc) return rc;
    MGR_HIP(hipStreamSynchronize(ctx->stream));
    int32_t errv = 0;
    MGR_HIP(hipMemcpy(&errv, ctx->err_flag, sizeof(int32_t), hipMemcpyDeviceToHost));
    if (errv) return ctx->fail(MGR_ERR_TRACE, "a ray pair ended off the boundary or an interior origin has an empty ray");
    ctx->J_set = true;
    return MGR_OK;
}

extern "C" int mgr_radiation_field_shape(mgr_ctx *ctx, int precision, int *waves_per_group, int *steps_per_chunk,
                                         int capacity, int *n_tried, int *tried_waves, int *tried_steps,
                                         float *tried_ms)
{
    if (!ctx) return MGR_ERR_ARGUMENT;
    if (precision != MGR_FP32 && precision != MGR_FP64) return ctx->fail(MGR_ERR_ARGUMENT, "bad precision");
    int pi = shape_of(ctx, precision);
    if (pi == 2 && (!ctx->masks_valid || ctx->rf_nwg[2] == 0) && ctx->rf_nwg[0] > 0) pi = 0;   // not known yet: the last one
    if (waves_per_group) *waves_per_group = ctx->rf_nwg[pi];
    if (steps_per_chunk) *steps_per_chunk = ctx->rf_ch[pi];
    const int n = (int)ctx->tune_log.size();
    if (n_tried) *n_tried = n;
    for (int i = 0; i < n && i < capacity; i++) {
        if (tried_waves) tried_waves[i] = ctx->tune_log[i].nwg;
        if (tried_steps) tried_steps[i] = ctx->tune_log[i].ch;
        if (tried_ms) tried_ms[i] = ctx->tune_log[i].ms;
    }
    return MGR_OK;
}

extern "C" int mgr_set_radiation_field_shape(mgr_ctx *ctx, int precision, int waves_per_group, int steps_per_chunk)
{
    if (!ctx) return MGR_ERR_ARGUMENT;
    if (precision != MGR_FP32 && precision != MGR_FP64) return ctx->fail(MGR_ERR_ARGUMENT, "bad precision");
    const bool fp64 = precision == MGR_FP64;
    const int pi = fp64 ? 1 : 0;
    if (waves_per_group == 0 && steps_per_chunk == 0) {
        ctx->rf_nwg[pi] = ctx->rf_ch[pi] = 0;   // the next radiation field tunes again
        if (!fp64) ctx->rf_nwg[2] = ctx->rf_ch[2] = 0;
    } else {
        const int chmax = fp64 ? max_chunk<double>(ctx) : max_chunk<float>(ctx);
        if (waves_per_group < 1 || waves_per_group > MAX_WAVES)
            return ctx->fail(MGR_ERR_ARGUMENT, "waves_per_group must be 1.." + std::to_string(MAX_WAVES));
        if (steps_per_chunk < 2 || steps_per_chunk > chmax)
            return ctx->fail(MGR_ERR_ARGUMENT, "steps_per_chunk must be 2.." + std::to_string(chmax) +
                                                   " for this model's line rows");
        const FieldLds lds = fp64 ? window_lds<double>(ctx, waves_per_group, steps_per_chunk)
                                  : window_lds<float>(ctx, waves_per_group, steps_per_chunk);
        if (lds.points < 2) return ctx->fail(MGR_ERR_UNSUPPORTED, "line rows do not fit the LDS budget");
        ctx->rf_nwg[pi] = waves_per_group;
        ctx->rf_ch[pi] = lds.points;
        if (!fp64) {
            ctx->rf_nwg[2] = waves_per_group;
            ctx->rf_ch[2] = steps_per_chunk;
        }
    }
    // the ALI graphs were captured with the previous shape
    if (ctx->graph_precision == precision) {
        MGR_HIP(hipSetDevice(ctx->device));
        if (ctx->graph_normal) (void)hipGraphExecDestroy(ctx->graph_normal);
        if (ctx->graph_ng) (void)hipGraphExecDestroy(ctx->graph_ng);
        ctx->graph_normal = ctx->graph_ng = nullptr;
        ctx->graph_precision = -1;
    }
    return MGR_OK;
}

extern "C" int mgr_compute_image(mgr_ctx *ctx, int64_t ray, int precision, double *I_m, double *I_p)
{
    if (!ctx) return MGR_ERR_ARGUMENT;
    if (precision != MGR_FP32 && precision != MGR_FP64) return ctx->fail(MGR_ERR_ARGUMENT, "precision must be MGR_FP32 or MGR_FP64");
    // sim_radiation.tpp:353-358
    if (!ctx->spectral_set || !ctx->spectral_image)
        return ctx->fail(MGR_ERR_STATE, "Spectral discretisation was not set for Images");
    if (!ctx->bdy_set) return ctx->fail(MGR_ERR_STATE, "compute_boundary_intensities first");
    if (!ctx->pops_set) return ctx->fail(MGR_ERR_STATE, "level populations not set");
    if (ctx->M != 1) return ctx->fail(MGR_ERR_UNSUPPORTED, "images are per model (batch of one)");
    if (ray < 0 || ray >= ctx->R / 2) return ctx->fail(MGR_ERR_ARGUMENT, "image ray must be in [0, nrays/2)");
    MGR_HIP(hipSetDevice(ctx->device));
    int rc = launch_trace_image(ctx, ray);
    if (rc) return rc;
    mgr_ctx::ImageTrace &g = ctx->img;
    const int64_t NF = ctx->N * ctx->F;
    if (!g.I_m) {
        MGR_HIP(device_malloc((void **)&g.I_m, NF * sizeof(double)));
        MGR_HIP(device_malloc((void **)&g.I_p, NF * sizeof(double)));
    }
    MGR_HIP(hipMemsetAsync(ctx->err_flag, 0, sizeof(int32_t), ctx->stream));
    rc = precision == MGR_FP64 ? launch_image<double>(ctx, ctx->row64) : launch_image<float>(ctx, ctx->row32);
    if (rc) return rc;
    MGR_HIP(hipStreamSynchronize(ctx->stream));
    int32_t errv = 0;
    MGR_HIP(hipMemcpy(&errv, ctx->err_flag, sizeof(int32_t), hipMemcpyDeviceToHost));
    if (errv) return ctx->fail(MGR_ERR_TRACE, "an image ray ended off the boundary or an interior origin has an empty ray");
    if (I_m && (rc = copy_to_host(ctx, I_m, g.I_m, NF * sizeof(double)))) return rc;
    if (I_p && (rc = copy_to_host(ctx, I_p, g.I_p, NF * sizeof(double)))) return rc;
    return MGR_OK;
}

// Radiation::u (radiation.cpp:117-126): with scattering every radiation
// field keeps each ray pair's u at the origin (sim_radiation.tpp:226-237,
// 258-262).  Allocates [R/2][N*F] doubles on the device; the ALI graphs are
// rebuilt so that they write it too.
extern "C" int mgr_set_scattering(mgr_ctx *ctx, int use_scattering)
{
    if (!ctx) return MGR_ERR_ARGUMENT;
    MGR_HIP(hipSetDevice(ctx->device));
    MGR_HIP(hipStreamSynchronize(ctx->stream));
    if (use_scattering && !ctx->u_store) {
        const size_t n = (size_t)(ctx->R / 2) * ctx->N * ctx->F;
        MGR_HIP(device_malloc((void **)&ctx->u_store, std::max<size_t>(n, 1) * sizeof(double)));
        MGR_HIP(hipMemset(ctx->u_store, 0, std::max<size_t>(n, 1) * sizeof(double)));
    } else if (!use_scattering && ctx->u_store) {
        (void)hipFree(ctx->u_store);
        ctx->u_store = nullptr;
    }
    ctx->graph_precision = -1;   // captured launches hold the old pointer
    return MGR_OK;
}

namespace mgr {

// Builds the far-end intensity cache of a precision when it is missing or
// stale (once per trace, frequency grid and boundary intensities).  It is
// skipped, and the kernel computes the intensities itself, when the cache and
// the spans would take more than three quarters of the device memory free
// without them, or an entry has no boundary cell at its far end (the kernel then reports that error).
int launch_far_cache(mgr_ctx *ctx, int precision)
{
    const int pi = precision == MGR_FP64 ? 1 : 0;
    if (!ctx->far_cache || ctx->far_valid[pi] || ctx->far_bad[pi] || !ctx->traced || !ctx->spectral_set ||
        !ctx->bdy_set)
        return MGR_OK;
    void **buf = pi ? (void **)&ctx->far_I64 : (void **)&ctx->far_I32;
    const size_t bytes = (size_t)ctx->NQ * (size_t)ctx->F * (pi ? sizeof(double) : sizeof(float));
    if (!*buf) {
        size_t fr = 0, tot = 0;
        const int64_t nspan = std::min<int64_t>((ctx->F + WAVE - 1) / WAVE, STEP_MASK_CHUNKS) *
                              ((ctx->span32 ? 1 : 0) + (ctx->span64 ? 1 : 0));
        const size_t spans = (size_t)(nspan * ctx->span_stride) * sizeof(uint16_t);
        if (hipMemGetInfo(&fr, &tot) != hipSuccess || !leaves_quarter(bytes, spans, fr + blocks_kept(ctx->device)) ||
            block_malloc(ctx->device, buf, std::max<size_t>(bytes, 8)) != hipSuccess) {
            (void)hipGetLastError();
            *buf = nullptr;
            ctx->far_bad[pi] = true;
            return MGR_OK;
        }
    }
    ctx->graph_precision = -1;   // captured launches may have read no cache, or a stale one
    RFArgs<float> a = RFArgs<float>();
    a.N = ctx->N;
    a.F = (int)ctx->F;
    a.cell_model = ctx->d_cell_model;
    a.cell_qbase = ctx->d_cell_qbase;
    a.m_R = ctx->d_m_R;
    a.nu = ctx->nu;
    a.cell2bdy = ctx->cell2bdy;
    a.I_bdy = ctx->I_bdy;
    a.far_cell = ctx->far_cell;
    a.far_shift = ctx->far_shift;
    // one wave per entry, four to a workgroup; a launch holds fewer than 2^32
    // threads, larger models' waves take several entries
    const int64_t entries = ctx->N * ctx->R;
    const dim3 grid((unsigned)std::min<int64_t>((entries + 3) / 4, 1 << 23));
    MGR_HIP(hipMemsetAsync(ctx->err_flag, 0, sizeof(int32_t), ctx->stream));
    if (pi)
        hipLaunchKernelGGL(k_far_cache<double>, grid, dim3(256), 0, ctx->stream, a, (int)ctx->R, ctx->far_I64,
                           ctx->err_flag);
    else
        hipLaunchKernelGGL(k_far_cache<float>, grid, dim3(256), 0, ctx->stream, a, (int)ctx->R, ctx->far_I32,
                           ctx->err_flag);
    MGR_LAUNCH_CHECK();
    int32_t errv = 0;
    MGR_HIP(hipStreamSynchronize(ctx->stream));
    MGR_HIP(hipMemcpy(&errv, ctx->err_flag, sizeof(int32_t), hipMemcpyDeviceToHost));
    if (errv) ctx->far_bad[pi] = true;
    else ctx->far_valid[pi] = true;
    return MGR_OK;
}

}  // namespace mgr

extern "C" int mgr_set_far_cache(mgr_ctx *ctx, int enable)
{
    if (!ctx) return MGR_ERR_ARGUMENT;
    MGR_HIP(hipSetDevice(ctx->device));
    MGR_HIP(hipStreamSynchronize(ctx->stream));
    ctx->far_cache = enable != 0;
    if (!ctx->far_cache) {
        free_far(ctx);
    }
    ctx->far_invalidate();
    ctx->graph_precision = -1;   // captured launches hold the old choice
    return MGR_OK;
}

extern "C" int mgr_set_window_skip(mgr_ctx *ctx, int enable)
{
    if (!ctx) return MGR_ERR_ARGUMENT;
    ctx->rf_window_skip = enable != 0;
    ctx->rf_spans = enable != 2;
    ctx->graph_precision = -1;   // captured launches hold the old choice
    return MGR_OK;
}

extern "C" int mgr_get_u(mgr_ctx *ctx, double *u)
{
    if (!ctx || !u) return MGR_ERR_ARGUMENT;
    if (!ctx->u_store) return ctx->fail(MGR_ERR_STATE, "scattering is off (mgr_set_scattering)");
    MGR_HIP(hipSetDevice(ctx->device));
    MGR_HIP(hipStreamSynchronize(ctx->stream));
    return copy_to_host(ctx, u, ctx->u_store, (size_t)(ctx->R / 2) * ctx->N * ctx->F * sizeof(double));
}
