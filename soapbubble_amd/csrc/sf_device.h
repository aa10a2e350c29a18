// Device-side data structures and helpers of the soap-film step for gfx950.
//
// Layout in HBM (packed over all bubbles of a context):
//   every cell field is one array; bubble b owns cells [off, off + nth*nph)
//   row-major by theta with phi contiguous, as the reference stores them
//   (quantity.cu:20-29). u_theta uses rows 0..nth-2 of its block; row nth-1
//   is padding that stays zero.
//   Per-row tables (nth+1 slots per bubble, base rt0) and per-column tables
//   (nph slots, base ct0) hold sin/cos of the cell coordinates in FP64 and
//   FP32, so no kernel evaluates the trigonometry of its own grid point.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sfk {

struct BubbleDev {
    int nth, nph, mask;          // nph = 2 nth; mask = nph - 1 when nph is a power of two, else -1
    int rt0, ct0, pr0;           // row-table, column-table and partial-sum bases
    long long off;               // first cell of this bubble in every cell field
    double h, invh, dt;          // grid spacing, 1/h, non-dimensional step
    double M, Cr, gs, gamma_max, eva;
    double re;                   // Re^-1 of the VISCOUS path
    // products of the row systems that hold for a whole bubble, in scalar
    // registers there: 1/dt, Cr dt, M dt / h^2
    double inv_dt, cr_dt, w_scale;
    float invh32, dt32;          // 1/h and dt for the FP32 traces
    double air_scale;            // radius / U: speed of the air corridor
    int gravity, evaporation, airflow, viscous;
};

// Air-flow time of one bubble (seconds) and its step in seconds; kernels
// derive the corridor factor 3 - |t - 3| and the mirror blend t/12. The
// update kernel marks a pending advance (when `advance`), which the next
// step's advection kernel applies before the assembly reads the time.
struct BubbleTime {
    double t;
    double dt_s;
    int advance;
    int pending;
    int nans;   // sticky: set once a NaN has been written into the state fields
    // initial guess of the Gamma solve: solves whose correction Gamma^{n+1} -
    // Gamma* is stored (0..2; the host resets it when the state or dt
    // changes), and the increment the update kernel leaves for the next
    // advection to apply
    int ghist;
    int gpend;
    // stop on a failed solve (the reference's `broken`, bubble.cu:1500-1507,
    // after which its frame loop takes no further step): bit 0 the option,
    // bit 1 set by the update kernel when this bubble's solve missed its
    // tolerance, bit 2 set by the next step's assembly. Kernels before the
    // assembly skip a bubble with bits 0 and 1, those after it one with bit
    // 2, so each launch reads a bit that an earlier launch wrote. Bit 3: the
    // captured steps wait for the host (StepGate); every kernel skips the bubble
    // until the host has taken the bit back.
    int stop;
};
constexpr int kPaused = 8;

__device__ __forceinline__ bool stopped_early(const BubbleTime& t) {
    return (t.stop & 3) == 3 || (t.stop & kPaused);
}
__device__ __forceinline__ bool stopped(const BubbleTime& t) { return (t.stop & (4 | kPaused)) != 0; }

// Per-bubble control block of the iterative solve. Every field is written by
// one kernel (the block of a row launch that arrives last, see arrive_last)
// and read only by later kernels of the same stream.
struct SolveCtl {
    double rz[2];        // r.z of inner iterations, slot = iteration parity
    double rr_in0;       // |r_in|^2 at the start of the current inner solve
    double rel_res;      // last relative (or absolute) residual, FP64
    double bb;           // |b|^2
    double mu;           // spectral bound of the line-preconditioned operator
    int outer_done;      // 1 once the FP64 residual met the tolerance
    int inner_done;      // 1 once the inner solve met its reduction
    int iters;           // inner iterations executed
    int outers;          // FP64 residual evaluations
    int xbuf;            // which x buffer holds the current iterate
    int converged;       // final verdict written by the finalize kernel
};

// Per-bubble history of the solves since creation (written by k_finalize).
struct SolveHist {
    int fails;
    int solves;
    double max_res;
};

// Statistics of the captured step for its inner-iteration schedule, since
// the host last cleared them: the largest tail ratio of the first
// refinement and the number of further refinements that ran.
struct SchedStat {
    double tail_ratio;
    int extra;
    int pad_;
};

// The gate of captured steps in the stiff regime, where the iterations a solve
// needs rest on the film: before the update of a step, k_gate looks at every
// bubble's residual and, with the spectral preconditioner, at its condition
// bound. A step that missed its tolerance or whose film is too uneven is not
// applied and no later one runs, until the host has taken that step itself.
struct StepGate {
    int done;     // steps applied since the host last opened the gate
    int why;      // kGateMissed, kGateUneven: what closed it (0: open)
    int accept;   // solves that miss their tolerance are applied
    int pad_;
};
constexpr int kGateMissed = 1, kGateUneven = 2;

struct Tables {
    // per-row, FP64: centres (j+1/2)h, faces j h (advection positions),
    // face sines of the assembly (pole faces exactly 0), csc of centres
    const double *sinTc, *cosTc, *sinTf, *cosTf, *sinFace, *cscTc;
    // per-row, FP32 copies
    const float *sinTc32, *cosTc32, *sinTf32, *cosTf32;
    // per-column: phi = i h
    const double *sinPc, *cosPc;
};

template <typename T> struct TabSel;
template <> struct TabSel<double> {
    static __device__ __forceinline__ double invh(const BubbleDev& B) { return B.invh; }
    static __device__ __forceinline__ double dt(const BubbleDev& B) { return B.dt; }
    static __device__ __forceinline__ const double* sTc(const Tables& t) { return t.sinTc; }
    static __device__ __forceinline__ const double* cTc(const Tables& t) { return t.cosTc; }
    static __device__ __forceinline__ const double* sTf(const Tables& t) { return t.sinTf; }
    static __device__ __forceinline__ const double* cTf(const Tables& t) { return t.cosTf; }
};
template <> struct TabSel<float> {
    static __device__ __forceinline__ float invh(const BubbleDev& B) { return B.invh32; }
    static __device__ __forceinline__ float dt(const BubbleDev& B) { return B.dt32; }
    static __device__ __forceinline__ const float* sTc(const Tables& t) { return t.sinTc32; }
    static __device__ __forceinline__ const float* cTc(const Tables& t) { return t.cosTc32; }
    static __device__ __forceinline__ const float* sTf(const Tables& t) { return t.sinTf32; }
    static __device__ __forceinline__ const float* cTf(const Tables& t) { return t.cosTf32; }
};

// ---------------------------------------------------------------- math ----
__device__ __forceinline__ float tfloor(float x) { return floorf(x); }
__device__ __forceinline__ double tfloor(double x) { return floor(x); }
// FP32: the hardware square root (within an ulp) without the
// correctly-rounded refinement sequence sqrtf expands to
__device__ __forceinline__ float tsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double tsqrt(double x) { return sqrt(x); }
__device__ __forceinline__ bool tisnan(float x) { return __builtin_isnan(x); }
__device__ __forceinline__ bool tisnan(double x) { return __builtin_isnan(x); }

// FP32 atan2 for the traced points: octant reduction to a = min/max in
// [0, 1] and atan(a) = a P(a^2), P of degree 8 fitted to atan(a)/a on [0, 1]
// by iteratively reweighted least squares on the relative error (Lawson's
// algorithm); maximum absolute error 1.2e-7 rad evaluated in FP32, i.e. a
// few 1e-5 of a cell at nTheta = 1024, below the FP32 resolution of the
// index-space position. FP64 keeps the library atan2.
__device__ __forceinline__ float tatan2(float y, float x) {
    const float ax = fabsf(x), ay = fabsf(y);
    const float mx = fmaxf(ax, ay), mn = fminf(ax, ay);
    const float a = mx > 0.0f ? mn * __builtin_amdgcn_rcpf(mx) : 0.0f;
    const float s = a * a;
    float p = 0.002850157907232642f;
    p = p * s - 0.01606966182589531f;
    p = p * s + 0.0426931269466877f;
    p = p * s - 0.07504424452781677f;
    p = p * s + 0.10640992224216461f;
    p = p * s - 0.1420365869998932f;
    p = p * s + 0.1999262124300003f;
    p = p * s - 0.3333307206630707f;
    p = p * s + 1.0f;
    float r = a * p;
    if (ay > ax) r = 1.57079632679489662f - r;
    if (x < 0.0f) r = 3.14159265358979324f - r;
    return copysignf(r, y);
}
__device__ __forceinline__ double tatan2(double y, double x) { return atan2(y, x); }

// 1 / sqrt(s) of a positive s: FP32 the hardware estimate (within an ulp);
// FP64 that estimate r (about 1e-8) times 1 + e/2 + 3 e^2/8, e = 1 - s r^2
// (the next term is below 1e-23), within an ulp or two.
__device__ __forceinline__ float inv_root(float s) { return __builtin_amdgcn_rsqf(s); }
__device__ __forceinline__ double inv_root(double s) {
    const double r = __builtin_amdgcn_rsq(s);
    const double e = fma(-(s * r), r, 1.0);
    return fma(r * e, fma(e, 0.375, 0.5), r);
}
// FP64 reciprocal of a positive finite y: the hardware estimate refined by
// two Newton steps r += r (1 - y r), each of which squares the relative
// error; the result is within an ulp or two of 1 / y.
__device__ __forceinline__ double rcp64(double y) {
    double r = __builtin_amdgcn_rcp(y);
    double e = fma(-y, r, 1.0);
    r = fma(r, e, r);
    e = fma(-y, r, 1.0);
    return fma(r, e, r);
}
// a / y through the refined reciprocal (within an ulp or two of the
// quotient, a quarter of the division's cost); a divisor of magnitude
// outside [1e-300, 1e300] (zero, denormal, huge, infinite or NaN) takes the
// division itself, so that 2 / 0 = inf and 0 / 0 = NaN come out as the
// reference's.
__device__ __forceinline__ double qdiv(double a, double y) {
    const double ay = fabs(y);
    if (ay >= 1e-300 && ay <= 1e300) return a * rcp64(y);
    return a / y;
}

__device__ __forceinline__ void tsincos(float x, float* s, float* c) { sincosf(x, s, c); }
__device__ __forceinline__ void tsincos(double x, double* s, double* c) { sincos(x, s, c); }
__device__ __forceinline__ float tfma(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double tfma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float tabs(float x) { return fabsf(x); }
__device__ __forceinline__ double tabs(double x) { return fabs(x); }
__device__ __forceinline__ float tmax(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double tmax(double a, double b) { return fmax(a, b); }
__device__ __forceinline__ float tmin(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ double tmin(double a, double b) { return fmin(a, b); }

// bubbleLerp (bubble.cu:153-160): NaN operands are skipped. With NANS =
// false the fields are known to hold no NaN (a per-bubble flag that every
// writer of a NaN sets) and the same expression is evaluated without the
// checks.
template <typename T>
__device__ __forceinline__ T lerp_nan(T from, T to, T alpha) {
    if (tisnan(from)) return to;
    if (tisnan(to)) return from;
    return (T(1) - alpha) * from + alpha * to;
}
template <typename T, bool NANS>
__device__ __forceinline__ T lerp_s(T from, T to, T alpha) {
    if (NANS) return lerp_nan(from, to, alpha);
    return (T(1) - alpha) * from + alpha * to;
}

// validateCoord (bubble.cu:116-137). The phi wrap fmod(y + nph, nph) is done
// by exact conditional subtraction (y + nph lies in [0, 3 nph) for every
// point the trace produces), which gives the same value as fmod.
template <typename T>
__device__ __forceinline__ bool validate_coord(T& x, T& y, int nth, int nph) {
    bool ret = false;
    const T tn = (T)nth, tp = (T)nph;
    if (x >= tn) { x = tp - x; y += tn; ret = !ret; }
    if (x < T(0)) { x = -x; y += tn; ret = !ret; }
    T a = y + tp;
    if (a >= T(2) * tp) a -= T(2) * tp;
    else if (a >= tp) a -= tp;
    y = a;
    return ret;
}

// A phi column x in [-nph, 2 nph) wrapped into the row: one AND for a row
// whose length is a power of two (mask = nph - 1); otherwise (mask = -1) a
// conditional add or subtract, clamped into the row so that no column,
// however malformed, addresses memory outside it.
__device__ __forceinline__ int wrap_col(int x, int nph, int mask) {
    if (mask >= 0) return x & mask;
    const int r = x < 0 ? x + nph : (x >= nph ? x - nph : x);
    return min(max(r, 0), nph - 1);
}

// Cell (j, i) of thread threadIdx.x in a packed tile {bubble, first row,
// first column, width}; tile widths are powers of two (a row shorter than
// its tile leaves the tile's last columns idle).
__device__ __forceinline__ void tile_cell(const int4& tl, int& j, int& i) {
    const int sh = __builtin_ctz((unsigned)tl.w);
    j = tl.y + ((int)threadIdx.x >> sh);
    i = tl.z + ((int)threadIdx.x & (tl.w - 1));
}

// A field of one bubble. P2 = true: the row length is known to be a power
// of two (mask = nph - 1), so the phi wrap is one AND; otherwise wrap_col
// takes the row's mask at run time.
template <typename T, bool P2 = false>
struct Field {
    const T* __restrict__ p;   // bubble base
    int nph, mask, maxrow;
    __device__ __forceinline__ int col(int c) const {
        if constexpr (P2) return c & mask;
        else return wrap_col(c, nph, mask);
    }
    __device__ __forceinline__ bool pow2() const { return P2 || mask >= 0; }
    // rows are clamped into the field so that no position, however
    // malformed, addresses memory outside it
    __device__ __forceinline__ T at(int row, int c) const {
        row = min(max(row, 0), maxrow);
        return p[(unsigned)(row * nph + col(c))];
    }
    template <bool NANS>
    __device__ __forceinline__ T belt(int row, int lo, T a) const {
        row = min(max(row, 0), maxrow);
        const T* r = p + (unsigned)(row * nph);
        return lerp_s<T, NANS>(r[col(lo)], r[col(lo + 1)], a);
    }
    __device__ __forceinline__ T belt(int row, int lo, T a) const { return belt<true>(row, lo, a); }
};

// ------------------------------------------------ interior fast path ----
// Away from the polar rows every sampler reduces to one bilinear
// interpolation between two adjacent rows with no reflection (validateCoord
// leaves theta alone, no pole branch applies). For fields without NaNs that
// case is evaluated directly, in both precisions and for rows of any length:
// byte offsets into a buffer resource, the next row through the scalar
// offset, a corner's two phi neighbours as one 8-byte (FP64: 16-byte) load.
// The pair of the row's last column takes its second value from the next
// row: that column loads column 0 instead (few lanes of few waves). Two
// loads an interpolation instead of four. A buffer load outside the field
// returns 0, so no position, however malformed, can read outside it; the
// resource of a field ends kFieldPad values after it (the last pair of its
// last row), which the state arrays are allocated with.
constexpr int kFieldPad = 4;
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t field_rsrc(const T* p, int cells) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0,
                                             (cells + kFieldPad) * (int)sizeof(T), 0x00020000);
}
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void bload1(__amdgpu_buffer_rsrc_t r, int off, int soff, float& v) {
    v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0));
}
__device__ __forceinline__ void bload1(__amdgpu_buffer_rsrc_t r, int off, int soff, double& v) {
    v = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
}
__device__ __forceinline__ void bload2(__amdgpu_buffer_rsrc_t r, int off, int soff, float& a,
                                       float& b) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0);
    a = __uint_as_float(v.x);
    b = __uint_as_float(v.y);
}
__device__ __forceinline__ void bload2(__amdgpu_buffer_rsrc_t r, int off, int soff, double& a,
                                       double& b) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0);
    u32x2 lo, hi;
    lo.x = v.x; lo.y = v.y; hi.x = v.z; hi.y = v.w;
    a = __builtin_bit_cast(double, lo);
    b = __builtin_bit_cast(double, hi);
}

// A traced position in index coordinates, x = ix + fx, y = iy + fy: the
// start point's integer index apart from the fraction, which holds the start
// point's half index and the increment turned along the circle. The
// interpolation weights then carry the increment's precision instead of the
// ulp of the absolute index (FP32: 6e-5 of a cell at index 1000).
template <typename T>
struct TPos {
    int ix, iy;
    T fx, fy;
    __device__ __forceinline__ T x() const { return (T)ix + fx; }
    __device__ __forceinline__ T y() const { return (T)iy + fy; }
};

// x split into its floor and the fraction above it.
__device__ __forceinline__ void split_floor(float x, int& i, float& f) {
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(i) : "v"(x));
    f = __builtin_amdgcn_fractf(x);
}
__device__ __forceinline__ void split_floor(double x, int& i, double& f) {
    const double fl = floor(x);
    i = (int)fl;
    f = x - fl;
}

// The lower corner of a sample point: row, column (wrapped into the row) and
// the weights above it.
template <typename T>
struct Corner {
    int t, c;
    T aT, aP;
};

// The corner of the point p + (OX, OY) / 2, added to the fraction exactly:
// weights from the fraction, row and column from the integer parts.
template <int OX, int OY, typename T, bool P2>
__device__ __forceinline__ Corner<T> corner_at(const TPos<T>& p, int nph, int mask) {
    Corner<T> q;
    split_floor(OX ? p.fx + T(0.5 * OX) : p.fx, q.t, q.aT);
    split_floor(OY ? p.fy + T(0.5 * OY) : p.fy, q.c, q.aP);
    q.t += p.ix;
    q.c += p.iy;
    q.c = P2 ? (q.c & mask) : wrap_col(q.c, nph, mask);
    return q;
}

// The lower row in [0, rows - 2]: no pole between the corners (rows: the
// field's row count).
template <typename T>
__device__ __forceinline__ bool inside(const Corner<T>& q, int rows) {
    return (unsigned)q.t < (unsigned)(rows - 1);
}

// The interpolation inside the field. The three interpolations as v0 + a (v1
// - v0): two operations each instead of the reference's three for (1 - a) v0
// + a v1, the same value within a rounding.
template <typename T>
__device__ __forceinline__ T corner_bilerp(__amdgpu_buffer_rsrc_t r, const Corner<T>& q, int nph) {
    const int rb = nph * (int)sizeof(T);
    const int row = __mul24(q.t, nph);
    const int off = (row + q.c) * (int)sizeof(T);
    T v00, v01, v10, v11;
    bload2(r, off, 0, v00, v01);
    bload2(r, off, rb, v10, v11);
    if (q.c == nph - 1) {
        bload1(r, row * (int)sizeof(T), 0, v01);
        bload1(r, row * (int)sizeof(T), rb, v11);
    }
    const T lo = tfma(q.aP, v01 - v00, v00);
    const T hi = tfma(q.aP, v11 - v10, v10);
    return tfma(q.aT, hi - lo, lo);
}

// The interpolation of a field of `rows` rows whose lower or upper row is
// the one across a pole: the field's first or last row at phi + pi, with the
// sign SIGN (values that flip across the pole); HALF (u_theta, whose rows
// stand a whole row from the pole): the two rows two apart, so the distance
// from the row on this side counts half. What the samplers below give for
// any point of the sphere, theta in [0, pi].
template <int SIGN, bool HALF, typename T, bool P2>
__device__ __forceinline__ T pole_bilerp(__amdgpu_buffer_rsrc_t r, Corner<T> q, int rows, int nph,
                                         int mask) {
    auto opposite = [&](int c) {
        return P2 ? ((c + (nph >> 1)) & mask) : wrap_col(c + nph / 2, nph, mask);
    };
    if (q.t < -1) { q.t = -1; q.aT = T(0); }
    if (q.t > rows - 1) { q.t = rows - 1; q.aT = T(1); }
    T w0 = T(1) - q.aT, w1 = q.aT;
    int c0 = q.c, c1 = q.c;
    if (q.t < 0) {
        c0 = opposite(q.c);
        w0 = (HALF ? T(0.5) : T(1)) * T(SIGN) * w0;
        if (HALF) w1 = T(0.5) + T(0.5) * w1;
    }
    if (q.t >= rows - 1) {
        c1 = opposite(q.c);
        w1 = (HALF ? T(0.5) : T(1)) * T(SIGN) * w1;
        if (HALF) w0 = T(0.5) + T(0.5) * w0;
    }
    const int r0 = max(q.t, 0) * nph, r1 = min(q.t + 1, rows - 1) * nph;
    auto at = [&](int row, int c) {
        T v;
        bload1(r, (row + (c == nph ? 0 : c)) * (int)sizeof(T), 0, v);
        return v;
    };
    const T l0 = at(r0, c0), l1 = at(r0, c0 + 1), h0 = at(r1, c1), h1 = at(r1, c1 + 1);
    return w0 * tfma(q.aP, l1 - l0, l0) + w1 * tfma(q.aP, h1 - h0, h0);
}

// Split a sample position into indices and weights; the phi index is
// clamped into range so a NaN position cannot address memory outside the
// field.
template <typename T>
__device__ __forceinline__ void split_index(T x, T y, int nph, int& tI, int& pI, T& aT, T& aP) {
    T fy = tfloor(y), fx = tfloor(x);
    aP = y - fy;
    aT = x - fx;
    pI = (int)fy;
    tI = (int)fx;
    if ((unsigned)pI >= (unsigned)nph) pI = pI < 0 ? 0 : nph - 1;
}

// sampleCentered (bubble.cu:320-376)
template <typename T, bool NANS = true, bool P2 = false>
__device__ __forceinline__ T sample_centered(const Field<T, P2>& f, int nth, T rx, T ry) {
    if constexpr (sizeof(T) == 8 && !NANS) {
        // FP64 fields without NaNs, away from the polar rows: the bilinear
        // interpolation of rows floor(x) and floor(x) + 1 that the general
        // branch below reduces to, the phi wrap on the integer column
        if (rx >= 0.5 && rx < (double)nth - 0.5 && f.pow2()) {
            const T x = rx - T(0.5), fx = tfloor(x), fy = tfloor(ry);
            const T aT = x - fx, aP = ry - fy;
            const int pI = (int)fy;
            const T* r0 = f.p + (size_t)(int)fx * f.nph;
            const T* r1 = r0 + f.nph;
            const int c0 = f.col(pI), c1 = f.col(pI + 1);
            const T lower = (T(1) - aP) * r0[c0] + aP * r0[c1];
            const T higher = (T(1) - aP) * r1[c0] + aP * r1[c1];
            return (T(1) - aT) * lower + aT * higher;
        }
    }
    T x = rx - T(0.5), y = ry;
    const int nph = f.nph;
    bool fl = validate_coord(x, y, nth, nph);
    int tI, pI; T aT, aP;
    split_index(x, y, nph, tI, pI, aT, aP);
    if (tI == 0 && fl) {
        T higher = f.template belt<NANS>(0, pI, aP);
        T lower = f.template belt<NANS>(0, pI + nph / 2, aP);
        return lerp_s<T, NANS>(lower, higher, aT);
    }
    if (fl) tI -= 1;
    if (tI == nth - 1) {
        T lower = f.template belt<NANS>(tI, pI, aP);
        T higher = f.template belt<NANS>(tI, pI + nph / 2, aP);
        return lerp_s<T, NANS>(lower, higher, aT);
    }
    T lower = f.template belt<NANS>(tI, pI, aP);
    T higher = f.template belt<NANS>(tI + 1, pI, aP);
    return lerp_s<T, NANS>(lower, higher, aT);
}

// sampleCentered of two fields at one point (the eta and Gamma samples of
// advectionAllCentered, bubble.cu:957-960) sharing the index computation.
template <typename T, bool NANS = true, bool P2 = false>
__device__ __forceinline__ void sample_centered2(const Field<T, P2>& f, const Field<T, P2>& g, int nth, T rx, T ry, T& of,
                                 T& og) {
    T x = rx - T(0.5), y = ry;
    const int nph = f.nph;
    bool fl = validate_coord(x, y, nth, nph);
    int tI, pI; T aT, aP;
    split_index(x, y, nph, tI, pI, aT, aP);
    int r0 = tI, r1 = tI + 1, c0 = pI, c1 = pI;
    if (tI == 0 && fl) {
        r0 = 0; r1 = 0; c0 = pI + nph / 2;
    } else {
        if (fl) tI -= 1;
        if (tI == nth - 1) { r0 = tI; r1 = tI; c1 = pI + nph / 2; }
        else { r0 = tI; r1 = tI + 1; }
    }
    of = lerp_s<T, NANS>(f.template belt<NANS>(r0, c0, aP), f.template belt<NANS>(r1, c1, aP), aT);
    og = lerp_s<T, NANS>(g.template belt<NANS>(r0, c0, aP), g.template belt<NANS>(r1, c1, aP), aT);
}

// sampleVPhi (bubble.cu:178-240): values taken across the pole flip sign.
template <typename T, bool NANS = true, bool P2 = false>
__device__ __forceinline__ T sample_vphi(const Field<T, P2>& f, int nth, T rx, T ry) {
    T x = rx - T(0.5), y = ry + T(0.5);
    const int nph = f.nph;
    bool fl = validate_coord(x, y, nth, nph);
    int tI, pI; T aT, aP;
    split_index(x, y, nph, tI, pI, aT, aP);
    if (tI == 0 && fl) {
        T higher = -f.template belt<NANS>(0, pI, aP);
        T lower = f.template belt<NANS>(0, pI + nph / 2, aP);
        return lerp_s<T, NANS>(lower, higher, aT);
    }
    if (fl) tI -= 1;
    if (tI == nth - 1) {
        T lower = f.template belt<NANS>(tI, pI, aP);
        T higher = -f.template belt<NANS>(tI, pI + nph / 2, aP);
        T v = lerp_s<T, NANS>(lower, higher, aT);
        return fl ? -v : v;
    }
    T lower = f.template belt<NANS>(tI, pI, aP);
    T higher = f.template belt<NANS>(tI + 1, pI, aP);
    T v = lerp_s<T, NANS>(lower, higher, aT);
    return fl ? -v : v;
}

// sampleVTheta (bubble.cu:247-313): u_theta has nth-1 rows; the polar caps
// interpolate between the first/last row and its phi+pi mirror with half
// weight. A sample exactly at theta = pi (which the reference reads past
// the array for) takes the south-cap branch.
template <typename T, bool NANS = true, bool P2 = false>
__device__ __forceinline__ T sample_vtheta(const Field<T, P2>& f, int nth, T rx, T ry) {
    T x = rx - T(1), y = ry;
    const int nph = f.nph;
    bool fl = validate_coord(x, y, nth, nph);
    int tI, pI; T aT, aP;
    split_index(x, y, nph, tI, pI, aT, aP);
    const T tn = (T)nth;
    if ((rx < T(0) && rx > T(-1)) || (rx > tn && rx < tn + T(1))) {
        tI -= 1;
        aT += T(1);
    } else if (rx >= tn + T(1) || rx <= T(-1)) {
        tI -= 2;
    }
    if (tI == 0 && fl && rx > T(-1)) {
        T higher = -f.template belt<NANS>(0, pI, aP);
        T lower = f.template belt<NANS>(0, pI + nph / 2, aP);
        return lerp_s<T, NANS>(lower, higher, T(0.5) * aT);
    }
    if (tI >= nth - 1 && !fl) { tI = nth - 2; aT = T(1); }
    if (tI == nth - 2) {
        T lower = f.template belt<NANS>(tI, pI, aP);
        T higher = -f.template belt<NANS>(tI, pI + nph / 2, aP);
        T v = lerp_s<T, NANS>(lower, higher, T(0.5) * aT);
        return fl ? -v : v;
    }
    T lower = f.template belt<NANS>(tI, pI, aP);
    T higher = f.template belt<NANS>(tI + 1, pI, aP);
    T v = lerp_s<T, NANS>(lower, higher, aT);
    return fl ? -v : v;
}

// The samplers at a traced position. NANS: the reference's NaN-skipping
// interpolation at the absolute position; without it (fields that hold no
// NaN) one bilinear interpolation from the split position.
template <typename T, bool NANS, bool P2>
__device__ __forceinline__ void sample_velocity(const Field<T, P2>& uth, const Field<T, P2>& uph,
                                                int nth, const TPos<T>& p, T& vt, T& vp) {
    if constexpr (NANS) {
        vt = sample_vtheta<T, true, P2>(uth, nth, p.x(), p.y());
        vp = sample_vphi<T, true, P2>(uph, nth, p.x(), p.y());
    } else {
        const int nph = uth.nph, m = uth.mask;
        const Corner<T> a = corner_at<-2, 0, T, P2>(p, nph, m);
        const Corner<T> b = corner_at<-1, 1, T, P2>(p, nph, m);
        const auto ra = field_rsrc(uth.p, (nth - 1) * nph), rp = field_rsrc(uph.p, nth * nph);
        if (inside(a, nth - 1) && inside(b, nth)) {
            vt = corner_bilerp(ra, a, nph);
            vp = corner_bilerp(rp, b, nph);
        } else {
            vt = pole_bilerp<-1, true, T, P2>(ra, a, nth - 1, nph, m);
            vp = pole_bilerp<-1, false, T, P2>(rp, b, nth, nph, m);
        }
    }
}
template <typename T, bool NANS, bool P2>
__device__ __forceinline__ void sample_centred_at(const Field<T, P2>& f, const Field<T, P2>& g, int nth,
                                                  const TPos<T>& p, T& of, T& og) {
    if constexpr (NANS) {
        sample_centered2<T, true, P2>(f, g, nth, p.x(), p.y(), of, og);
    } else {
        const int nph = f.nph, m = f.mask;
        const Corner<T> q = corner_at<-1, 0, T, P2>(p, nph, m);
        const auto rf = field_rsrc(f.p, nth * nph), rg = field_rsrc(g.p, nth * nph);
        if (inside(q, nth)) {
            of = corner_bilerp(rf, q, nph);
            og = corner_bilerp(rg, q, nph);
        } else {
            of = pole_bilerp<1, false, T, P2>(rf, q, nth, nph, m);
            og = pole_bilerp<1, false, T, P2>(rg, q, nth, nph, m);
        }
    }
}

// ------------------------------------------------------ great circle ----
// One leg of a back-trace (traceGreatCircle, bubble.cu:416-506, and the
// vector advection kernels, bubble.cu:651-766, 787-902), in the coordinates
// of the start point: x towards its meridian's point of the equator, y east,
// z the pole, so the start point is w = (sin t0, 0, cos t0), its frame e_theta
// = (cos t0, 0, -sin t0), e_phi = (0, 1, 0), and no trigonometry of phi enters.
// Moving by `step` against the velocity (a, b) reaches
//   q = w cos(s) + (a e_theta + b e_phi) k,   s = |u| step, k = -step sin(s) / s,
// with sin(s) / s and cos(s) by their series in s^2 (no root of |u|^2, no
// unit direction). Its angles from the start point are
//   sin dphi   = q_y / rho,
//   sin dtheta = rho cos t0 - q_z sin t0 = a k + cos t0 q_y tan(dphi / 2)
// (the second form free of the first one's cancellation: it keeps the
// increment's relative precision in FP32). The velocity sampled at q is
// carried back along the circle by v - (v . w)(q + w) / (1 + q . w), in the
// two points' frames a rotation by g with
//   cos g (1 + cos s) = cos dphi (1 + q_z cos t0) + rho sin t0,
//   sin g (1 + cos s) = sin dphi (q_z + cos t0).
// The reference forms the same points and components from Cartesian
// vectors, a unit direction and its cross products: about 340 vector
// instructions a velocity trace, this form about 170.
template <typename T>
struct TraceStart {
    int ix, iy;
    T hx, hy;      // index coordinates ix + hx, iy + hy (hx, hy 0 or 1/2)
    T sT, cT;      // sin, cos of the start point's theta
};
template <typename T>
struct Leg {
    TPos<T> p;     // the point reached
    T cg, sg;      // rotation of its frame's components into the start frame's
};

// sin(s) / s, cos(s) and 1 / (1 + cos(s)) = sec^2(s/2) / 2 from s^2 below
// 1/256, truncated below the rounding (first term left out: s^6 / 7! =
// 1e-11, s^6 / 6!, 17 s^6 / 5760 = 2e-10 in FP32; s^12 / 13! and the like in
// FP64, the third through the reciprocal).
__device__ __forceinline__ void small_step(float s2, float& sc, float& c, float& in) {
    sc = fmaf(s2, fmaf(s2, 1.0f / 120.0f, -1.0f / 6.0f), 1.0f);
    c = fmaf(s2, fmaf(s2, 1.0f / 24.0f, -0.5f), 1.0f);
    in = fmaf(s2, fmaf(s2, 1.0f / 48.0f, 0.125f), 0.5f);
}
__device__ __forceinline__ void small_step(double s2, double& sc, double& c, double& in) {
    sc = 1.0 + s2 * (-1.0 / 6 + s2 * (1.0 / 120 + s2 * (-1.0 / 5040 + s2 * (1.0 / 362880 +
                                                                           s2 * (-1.0 / 39916800)))));
    c = 1.0 + s2 * (-0.5 + s2 * (1.0 / 24 + s2 * (-1.0 / 720 + s2 * (1.0 / 40320 +
                                                                     s2 * (-1.0 / 3628800)))));
    in = rcp64(1.0 + c);
}
// asin(s) and tan(asin(s) / 2) = s / (1 + sqrt(1 - s^2)) for |s| below 0.1
// (FP64: 0.063), cos(asin(s)) above CosMin: by their series (truncated at
// 5e-9 rad and 4e-8 relative in FP32; at 1e-19 in FP64, the second through
// the cosine)
template <typename T> struct CosMin;
template <> struct CosMin<float> { static constexpr float v = 0.995f; };
template <> struct CosMin<double> { static constexpr double v = 0.998; };
__device__ __forceinline__ float asin_small(float s) {
    const float s2 = s * s;
    return s * fmaf(s2, fmaf(s2, 3.0f / 40.0f, 1.0f / 6.0f), 1.0f);
}
__device__ __forceinline__ double asin_small(double s) {
    const double s2 = s * s;
    return s * (1.0 + s2 * (1.0 / 6 + s2 * (3.0 / 40 + s2 * (5.0 / 112 + s2 * (35.0 / 1152 +
                                                              s2 * (63.0 / 2816 + s2 * (231.0 / 13312)))))));
}
__device__ __forceinline__ float tan_half(float s, float) {
    const float y = s * s;
    return s * fmaf(y, fmaf(y, 0.0625f, 0.125f), 0.5f);
}
__device__ __forceinline__ double tan_half(double s, double c) { return s * rcp64(1.0 + c); }

template <typename T>
__device__ __forceinline__ void trace_leg(const TraceStart<T>& o, T a, T b, T step, T invh,
                                          Leg<T>& g) {
    const T s2 = tfma(a, a, b * b) * (step * step);
    T sc, c, in;
    small_step(s2, sc, c, in);
    const T k = -step * sc;
    T qx, qy = b * k, qz, rho, ir;
    const T ak = a * k;
    qx = tfma(o.cT, ak, o.sT * c);
    qz = tfma(-o.sT, ak, o.cT * c);
    const T r2 = tfma(qx, qx, qy * qy);
    ir = inv_root(r2);
    rho = r2 * ir;
    T sf = qy * ir, cf = qx * ir;
    T dth = asin_small(tfma(o.cT * qy, tan_half(sf, cf), ak)), dph = asin_small(sf);
    g.cg = tfma(cf, tfma(qz, o.cT, T(1)), rho * o.sT) * in;
    g.sg = sf * (qz + o.cT) * in;
    // cos dphi above CosMin bounds |sin dphi|, and s below 1/16 leaves
    // |sin dtheta| <= s + s |tan(dphi / 2)| < 0.066
    if (!(s2 < T(1.0 / 256) && cf > CosMin<T>::v)) {
        // a large step, or a trace that passes close to a pole: the same
        // angles by atan2, and the rotation from the tangents of the circle
        // at both points (1 + cos(s) loses its digits near the antipode)
        const T un = tsqrt(tfma(a, a, b * b)), iu = un > T(0) ? T(1) / un : T(0);
        const T ua = a * iu, ub = b * iu;
        T sn;
        tsincos(-un * step, &sn, &c);
        qx = tfma(o.cT * ua, sn, o.sT * c);
        qy = ub * sn;
        qz = tfma(-(o.sT * ua), sn, o.cT * c);
        rho = tsqrt(tfma(qx, qx, qy * qy));
        cf = T(1);    // at a pole: the start point's meridian
        sf = T(0);
        if (rho > T(0)) {
            cf = qx / rho;
            sf = qy / rho;
        }
        dth = tatan2(rho * o.cT - qz * o.sT, qz * o.cT + rho * o.sT);
        dph = tatan2(sf, cf);
        const T t0 = o.cT * ua * c - o.sT * sn, t1 = ub * c, t2 = -(o.sT * ua) * c - o.cT * sn;
        const T et = qz * (cf * t0 + sf * t1) - rho * t2, ep = cf * t1 - sf * t0;
        g.cg = et * ua + ep * ub;
        g.sg = et * ub - ep * ua;
    }
    g.p.ix = o.ix;
    g.p.iy = o.iy;
    g.p.fx = tfma(dth, invh, o.hx);
    g.p.fy = tfma(dph, invh, o.hy);
}

// A velocity (vt, vp) at the leg's point, in the start point's frame.
template <typename T>
__device__ __forceinline__ void carry_back(const Leg<T>& g, T vt, T vp, T& a, T& b) {
    a = tfma(vt, g.cg, -(vp * g.sg));
    b = tfma(vt, g.sg, vp * g.cg);
}

// The back-trace from a start point with velocity (a, b): the half step's
// velocity carried back, the full step with it. Returns whether the point
// moves (the reference returns the start point, and a zero or NaN speed for
// the velocity, where either speed is not positive); `speed2` that speed
// squared where it does not.
template <typename T, bool NANS, bool P2>
__device__ __forceinline__ bool back_trace(const Field<T, P2>& uth, const Field<T, P2>& uph, int nth,
                                           const TraceStart<T>& o, T a, T b, T dt, T invh, Leg<T>& g,
                                           T& speed2) {
    speed2 = a * a + b * b;
    bool moves = speed2 > T(0);
    if (moves) {
        T vt, vp;
        trace_leg(o, a, b, T(0.5) * dt, invh, g);
        sample_velocity<T, NANS, P2>(uth, uph, nth, g.p, vt, vp);
        carry_back(g, vt, vp, a, b);
        speed2 = a * a + b * b;
        moves = speed2 > T(0);
        if (moves) trace_leg(o, a, b, dt, invh, g);
    }
    if (!moves) g.p = TPos<T>{o.ix, o.iy, o.hx, o.hy};
    return moves;
}

// ------------------------------------------------------------ BIMOCQ ----
// Mapping arithmetic of the BIMOCQ scalar advection, FP64 in every precision
// mode. The reference keeps a map as index-space (theta, phi) pairs and
// converts every corner to a unit vector inside each spherical
// interpolation (lerpCoords, bubble.cu:512-536), and the result back. Here a
// map holds the unit vectors themselves: the interpolations chain on unit
// vectors, and only a position that samples a field is converted to index
// coordinates (acos of z, atan2 of y, x, as lerpCoords ends). The same
// arithmetic up to rounding, without two sin/cos pairs and an acos/atan2 per
// interpolation.
struct U3 {
    double x, y, z;
};
struct UMap {
    double *x, *y, *z;
};

__device__ __forceinline__ double safe_acos_d(double x) { return acos(fmax(-1.0, fmin(1.0, x))); }

__device__ __forceinline__ U3 unit_of_index(double h, double t, double f) {
    double st, ct, sf, cf;
    sincos(t * h, &st, &ct);
    sincos(f * h, &sf, &cf);
    return U3{cf * st, sf * st, ct};
}

struct P2d {
    double x, y;   // (theta, phi) index coordinates
};

// Index coordinates (acos z, atan2(y, x)) / h of a unit vector a few cells
// from the centre of cell (j, i): the centre's index coordinates (j + 1/2, i)
// plus the angles turned from it, each the asin of a sine that the (sin, cos)
// pair of the meridian half-plane (a unit vector) or the equatorial plane
// (scale rho) gives, by its series below 1/4; farther points take atan2. The
// same angles up to rounding, phi in the centre's period rather than atan2's
// (-pi, pi] (the samplers wrap phi either way).
struct CellRef {
    double gx, gy, sT, cT, sP, cP;
};
__device__ __forceinline__ CellRef cell_ref(const Tables& tab, const BubbleDev& B, int j, int i) {
    return CellRef{j + 0.5, (double)i, tab.sinTc[B.rt0 + j], tab.cosTc[B.rt0 + j],
                   tab.sinPc[B.ct0 + i], tab.cosPc[B.ct0 + i]};
}
// asin(s) for |s| < kAsinWide by its odd series (truncated at 2e-18)
constexpr double kAsinWide = 0.25;
__device__ __forceinline__ double asin_wide(double s) {
    const double y = s * s;
    double p = 676039.0 / 104857600.0;
    p = fma(p, y, 88179.0 / 12058624.0);
    p = fma(p, y, 46189.0 / 5505024.0);
    p = fma(p, y, 12155.0 / 1245184.0);
    p = fma(p, y, 6435.0 / 557056.0);
    p = fma(p, y, 143.0 / 10240.0);
    p = fma(p, y, 231.0 / 13312.0);
    p = fma(p, y, 63.0 / 2816.0);
    p = fma(p, y, 35.0 / 1152.0);
    p = fma(p, y, 5.0 / 112.0);
    p = fma(p, y, 3.0 / 40.0);
    p = fma(p, y, 1.0 / 6.0);
    return s * fma(p, y, 1.0);
}
__device__ __forceinline__ P2d index_near(double invh, const U3& r, const CellRef& o) {
    const double r2 = r.x * r.x + r.y * r.y;
    const double ir = inv_root(r2), rho = r2 * ir;
    const double nt = rho * o.cT - r.z * o.sT, ct = r.z * o.cT + rho * o.sT;
    const double np = (r.y * o.cP - r.x * o.sP) * ir, cp = r.x * o.cP + r.y * o.sP;
    P2d q;
    q.x = o.gx + asin_wide(nt) * invh;
    q.y = o.gy + asin_wide(np) * invh;
    if (!(ct > 0.0 && fabs(nt) < kAsinWide && cp > 0.0 && fabs(np) < kAsinWide)) {
        // (next to a pole, where phi turns far at once, the arc cosine of z
        // would leave theta a rounding of z over sin(theta))
        q.x = atan2(sqrt(r2), r.z) * invh;
        q.y = atan2(r.y, r.x) * invh;
    }
    return q;
}

// lerpCoords on unit vectors: the point a fraction alpha along the great
// circle from f to t (Rodrigues rotation about k = f x t / |f x t|); f when
// the two coincide (k undefined), as the reference returns `from`.
// Map values at neighbouring grid points are a few cells apart, so the angle
// theta between f and t is small: below |t - f| = 0.02 the rotation is the
// same point written as a f + b t with a = sin((1 - alpha) theta) / sin theta,
// b = sin(alpha theta) / sin theta, both by their series in theta^2, and
// theta^2 = (2 asin(|t - f| / 2))^2 by its series in |t - f|^2 (every
// truncation below 1e-16 relative there): no square root, division or
// normalisation. Larger angles rotate with acos and sincos.
__device__ __forceinline__ double slerp_coef(double beta, double u) {
    const double b2 = beta * beta;
    return beta * (1.0 + u * (1.0 - b2) *
                             (1.0 / 6 + u * ((7.0 - 3.0 * b2) / 360 +
                                             u * (31.0 + b2 * (-18.0 + 3.0 * b2)) / 15120)));
}
__device__ __forceinline__ U3 slerp_u(const U3& f, const U3& t, double alpha) {
    const double dx = t.x - f.x, dy = t.y - f.y, dz = t.z - f.z;
    const double d2 = dx * dx + dy * dy + dz * dz;
    if (d2 < 4e-4) {
        if (d2 == 0.0) return f;
        const double u = d2 * (1.0 + d2 * (1.0 / 12 + d2 * (1.0 / 90 + d2 * (1.0 / 560))));
        const double a = slerp_coef(1.0 - alpha, u), b = slerp_coef(alpha, u);
        return U3{a * f.x + b * t.x, a * f.y + b * t.y, a * f.z + b * t.z};
    }
    double kx = f.y * t.z - f.z * t.y, ky = f.z * t.x - f.x * t.z, kz = f.x * t.y - f.y * t.x;
    const double k2 = kx * kx + ky * ky + kz * kz;
    const double kin = 1.0 / sqrt(k2);
    kx *= kin; ky *= kin; kz *= kin;
    if (__builtin_isnan(kx)) return f;
    const double cth = f.x * t.x + f.y * t.y + f.z * t.z;
    double sn, cs;
    const double span = safe_acos_d(cth) * alpha;
    sincos(span, &sn, &cs);
    const double kf = kx * f.x + ky * f.y + kz * f.z;
    const double cx = ky * f.z - kz * f.y, cy = kz * f.x - kx * f.z, cz = kx * f.y - ky * f.x;
    return U3{f.x * cs + cx * sn + kx * kf * (1 - cs), f.y * cs + cy * sn + ky * kf * (1 - cs),
              f.z * cs + cz * sn + kz * kf * (1 - cs)};
}

// sampleMapping (bubble.cu:539-603) on a unit-vector map: the corner
// selection of the reference, three spherical interpolations.
__device__ __forceinline__ U3 sample_map_u(const UMap& M, size_t off, int nth, int nph, double rx, double ry) {
    const int m = (nph & (nph - 1)) == 0 ? nph - 1 : -1;
    if (rx >= 0.5 && rx < (double)nth - 0.5 && m >= 0) {
        // away from the polar rows: the corners of rows floor(x), floor(x) + 1
        // that the general branch below selects there, the phi wrap on the
        // integer column
        const double x = rx - 0.5, fx = floor(x), fy = floor(ry);
        const double aT = x - fx, aP = ry - fy;
        const int pI = (int)fy;
        const size_t r0 = off + (size_t)(int)fx * nph, r1 = r0 + nph;
        const size_t c0 = (size_t)(pI & m), c1 = (size_t)((pI + 1) & m);
        auto at = [&](size_t c) { return U3{M.x[c], M.y[c], M.z[c]}; };
        return slerp_u(slerp_u(at(r0 + c0), at(r0 + c1), aP), slerp_u(at(r1 + c0), at(r1 + c1), aP),
                       aT);
    }
    double x = rx - 0.5, y = ry;
    const bool fl = validate_coord(x, y, nth, nph);
    int pI = (int)floor(y), tI = (int)floor(x);
    const double aP = y - pI, aT = x - tI;
    if ((unsigned)pI >= (unsigned)nph) pI = pI < 0 ? 0 : nph - 1;
    auto at = [&](int row, int col) {
        row = min(max(row, 0), nth - 1);
        const size_t c = off + (size_t)row * nph + wrap_col(col, nph, m);
        return U3{M.x[c], M.y[c], M.z[c]};
    };
    U3 ll{0, 0, 1}, lr{0, 0, 1}, hl{0, 0, 1}, hr{0, 0, 1};
    if (fl) {
        if (tI == 0) {
            hl = at(0, pI); hr = at(0, pI + 1);
            ll = at(0, pI + nph / 2); lr = at(0, pI + 1 + nph / 2);
        } else {
            tI -= 1;
        }
    }
    if (tI == nth - 1) {
        ll = at(tI, pI); lr = at(tI, pI + 1);
        hl = at(tI, pI + nph / 2); hr = at(tI, pI + 1 + nph / 2);
    } else if (tI != 0 || !fl) {
        ll = at(tI, pI); lr = at(tI, pI + 1);
        hl = at(tI + 1, pI); hr = at(tI + 1, pI + 1);
    }
    return slerp_u(slerp_u(ll, lr, aP), slerp_u(hl, hr, aP), aT);
}

// The same interpolations where every pair is near (|t - f|^2 below
// kNearD2, grids of about 50 rows and more), for rows of any length; a row
// past a pole is the first or last one at phi + pi. The coefficients of the end a fraction
// beta away, sin(beta theta) / sin theta = beta (1 + u p1 + u^2 p2 + ...), u
// = theta^2, are polynomials in beta^2: formed once for the two
// interpolations along phi, and constants for the fixed sample points. One
// more term of each series than slerp_u's (truncated below 1e-16 at kNearD2).
constexpr double kNearD2 = 4e-3;
struct SlerpEnd {
    double k, p1, p2, p3, p4;
};
__device__ __forceinline__ constexpr SlerpEnd slerp_end(double beta) {
    const double b = beta * beta, q = 1.0 - b;
    return SlerpEnd{beta, q * (1.0 / 6), q * (7.0 / 360 - b * (1.0 / 120)),
                    q * (31.0 / 15120 + b * (-1.0 / 840 + b * (1.0 / 5040))),
                    q * (127.0 / 604800 + b * (-239.0 / 1814400 + b * (11.0 / 362880 - b / 362880)))};
}
__device__ __forceinline__ double slerp_weight(const SlerpEnd& e, double u) {
    return e.k * fma(u, fma(u, fma(u, fma(u, e.p4, e.p3), e.p2), e.p1), 1.0);
}
// `near` stays set while the pairs are near.
__device__ __forceinline__ U3 slerp_near(const U3& f, const U3& t, const SlerpEnd& ef,
                                         const SlerpEnd& et, bool& near) {
    const double dx = t.x - f.x, dy = t.y - f.y, dz = t.z - f.z;
    const double d2 = fma(dx, dx, fma(dy, dy, dz * dz));
    near = near && d2 < kNearD2;
    const double u =
        d2 * fma(d2, fma(d2, fma(d2, fma(d2, 1.0 / 3150, 1.0 / 560), 1.0 / 90), 1.0 / 12), 1.0);
    const double a = slerp_weight(ef, u), b = slerp_weight(et, u);
    return U3{fma(a, f.x, b * t.x), fma(a, f.y, b * t.y), fma(a, f.z, b * t.z)};
}
__device__ __forceinline__ U3 map_at(const UMap& M, size_t c) { return U3{M.x[c], M.y[c], M.z[c]}; }

// Row r (-1 .. nth) of a map: its first cell, and the columns to add.
__device__ __forceinline__ size_t map_row(const BubbleDev& B, size_t off, int r, int& shift) {
    shift = r < 0 || r >= B.nth ? B.nth : 0;
    return off + (size_t)min(max(r, 0), B.nth - 1) * B.nph;
}
// c in [0, 2 nph) wrapped into the row
__device__ __forceinline__ int fold_col(const BubbleDev& B, int c) {
    return c >= B.nph ? c - B.nph : c;
}

// sampleMapping at an index position (x, y); clears `near` where the general
// form is needed (its value is then meaningless).
__device__ __forceinline__ U3 sample_map_near(const UMap& M, size_t off, const BubbleDev& B, double rx,
                                              double ry, bool& near) {
    int tI, pI;
    double aT, aP;
    split_floor(rx - 0.5, tI, aT);
    split_floor(ry, pI, aP);
    near = near && tI >= -1 && tI < B.nth;
    tI = min(max(tI, -1), B.nth - 1);
    int sl, sh;
    const size_t r0 = map_row(B, off, tI, sl), r1 = map_row(B, off, tI + 1, sh);
    const int c = wrap_col(pI, B.nph, B.mask);
    const SlerpEnd f = slerp_end(1.0 - aP), t = slerp_end(aP);
    const U3 lo = slerp_near(map_at(M, r0 + fold_col(B, c + sl)),
                             map_at(M, r0 + fold_col(B, fold_col(B, c + 1) + sl)), f, t, near);
    const U3 hi = slerp_near(map_at(M, r1 + fold_col(B, c + sh)),
                             map_at(M, r1 + fold_col(B, fold_col(B, c + 1) + sh)), f, t, near);
    return slerp_near(lo, hi, slerp_end(1.0 - aT), slerp_end(aT), near);
}

// sampleMapping at the four quarter points around the centre of cell (j, i),
// in kMsDx / kMsDy order, and the centre itself (the map's own value): six
// interpolations along phi in three rows and four along theta, where five
// separate lookups make fifteen.
struct Around {
    U3 nw, sw, ne, se, mid;
};
__device__ __forceinline__ void sample_map_around(const UMap& M, size_t off, const BubbleDev& B, int j,
                                                  int i, Around& out, bool& near) {
    const int iw = i == 0 ? B.nph - 1 : i - 1, ie = i + 1 == B.nph ? 0 : i + 1;
    constexpr SlerpEnd q1 = slerp_end(0.25), q3 = slerp_end(0.75);
    U3 w[3], e[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        int sh;
        const size_t row = map_row(B, off, j - 1 + r, sh);
        const U3 c = map_at(M, row + fold_col(B, i + sh));
        w[r] = slerp_near(map_at(M, row + fold_col(B, iw + sh)), c, q1, q3, near);
        e[r] = slerp_near(c, map_at(M, row + fold_col(B, ie + sh)), q3, q1, near);
        if (r == 1) out.mid = c;
    }
    out.nw = slerp_near(w[0], w[1], q1, q3, near);
    out.sw = slerp_near(w[1], w[2], q3, q1, near);
    out.ne = slerp_near(e[0], e[1], q1, q3, near);
    out.se = slerp_near(e[1], e[2], q3, q1, near);
}
// the sample of kMsDx / kMsDy's number q (uniform)
__device__ __forceinline__ U3 pick(const Around& v, int q) {
    // (values, not references: the five stay in registers)
    auto sel = [q](double a, double b, double c, double d, double e) {
        return q == 0 ? +a : q == 1 ? +b : q == 2 ? +c : q == 3 ? +d : +e;
    };
    return U3{sel(v.nw.x, v.sw.x, v.ne.x, v.se.x, v.mid.x), sel(v.nw.y, v.sw.y, v.ne.y, v.se.y, v.mid.y),
              sel(v.nw.z, v.sw.z, v.ne.z, v.se.z, v.mid.z)};
}

// sampleCentered of a field without NaNs at an index position of a map.
__device__ __forceinline__ Corner<double> corner_of(const BubbleDev& B, const P2d& p) {
    Corner<double> q;
    split_floor(p.x - 0.5, q.t, q.aT);
    split_floor(p.y, q.c, q.aP);
    q.c = wrap_col(q.c, B.nph, B.mask);
    return q;
}
__device__ __forceinline__ double sample_corner(const double* f, const BubbleDev& B,
                                                const Corner<double>& q) {
    const auto r = field_rsrc(f, B.nth * B.nph);
    if (inside(q, B.nth)) return corner_bilerp(r, q, B.nph);
    return pole_bilerp<1, false, double, false>(r, q, B.nth, B.nph, B.mask);
}

// MULTISAMPLE (header.cuh:98): five samples around a point with these
// weights and offsets (bubble.cu:983-995)
__constant__ const double kMsW[5] = {0.125, 0.125, 0.125, 0.125, 0.5};
__constant__ const double kMsDx[5] = {-0.25, 0.25, -0.25, 0.25, 0.0};
__constant__ const double kMsDy[5] = {-0.25, -0.25, 0.25, 0.25, 0.0};

// -------------------------------------------------------- reductions ----
// Wave reductions by DPP (row shifts, then the last lanes of rows 0 and 2
// into the rows after them, of row 1 into rows 2 and 3): lane 63 holds the
// result, which every lane receives. Register moves a few cycles apart, where
// shuffles through the LDS unit wait a hundred for each of six levels: 0.3-0.5
// us a row kernel, which at the small sizes is one chain of latencies.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero(double v) {
    u32x2 u = __builtin_bit_cast(u32x2, v);
    const unsigned int x = u.x, y = u.y;
    u.x = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, false);
    u.y = (unsigned int)__builtin_amdgcn_update_dpp(0, (int)y, CTRL, ROWS, 0xf, false);
    return __builtin_bit_cast(double, u);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_or_zero(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ double last_lane(double v) {
    u32x2 u = __builtin_bit_cast(u32x2, v);
    const unsigned int x = u.x, y = u.y;
    u.x = (unsigned int)__builtin_amdgcn_readlane((int)x, 63);
    u.y = (unsigned int)__builtin_amdgcn_readlane((int)y, 63);
    return __builtin_bit_cast(double, u);
}
__device__ __forceinline__ float last_lane(float v) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
// `op` combines two values; a lane without a source combines with zero
template <typename T, typename Op>
__device__ __forceinline__ T wave_reduce(T v, Op op) {
    v = op(v, dpp_or_zero<0x111, 0xf>(v));   // row_shr:1
    v = op(v, dpp_or_zero<0x112, 0xf>(v));   // row_shr:2
    v = op(v, dpp_or_zero<0x114, 0xf>(v));   // row_shr:4
    v = op(v, dpp_or_zero<0x118, 0xf>(v));   // row_shr:8
    v = op(v, dpp_or_zero<0x142, 0xa>(v));   // row_bcast:15 into rows 1 and 3
    v = op(v, dpp_or_zero<0x143, 0xc>(v));   // row_bcast:31 into rows 2 and 3
    return last_lane(v);
}
__device__ __forceinline__ double wave_sum(double v) {
    return wave_reduce(v, [](double a, double b) { return a + b; });
}
// the maximum of non-negative values
__device__ __forceinline__ double wave_max(double v) {
    return wave_reduce(v, [](double a, double b) { return fmax(a, b); });
}
__device__ __forceinline__ float wave_max(float v) {
    return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}

// Deterministic block sum of NV values; every thread receives the sums.
// `red` must hold 16 * NV doubles of LDS.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* red) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
    __syncthreads();
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) red[k * 16 + wid] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double s = 0.0;
        for (int w = 0; w < nw; ++w) s += red[k * 16 + w];
        v[k] = s;
    }
    __syncthreads();
}

// Deterministic block maximum of a non-negative value; every thread receives
// it. `red` must hold 16 doubles of LDS.
__device__ __forceinline__ double block_max(double v, double* red) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    v = wave_max(v);
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double m = 0.0;
    for (int w = 0; w < nw; ++w) m = fmax(m, red[w]);
    __syncthreads();
    return m;
}

// The rows of a row block. A row of R threads (C cells each) takes R rounded
// up to whole waves; a block of at least twice that holds blockDim.x / w
// rows j0, j0 + 1, ... (packed: rows of several widths share one launch),
// one segment of w threads each; otherwise its one row has the whole block.
// seg: this thread's row (j0 + seg), lt: its place in the row, nt: threads a
// segment, nseg: segments of the block.
struct RowSeg {
    int seg, lt, nt, nseg;
};
// PACKED = false: the launch has one row a block (compiled to constants).
template <bool PACKED = true>
__device__ __forceinline__ RowSeg row_seg(int R) {
    const int w = (R + 63) & ~63;
    RowSeg s;
    if (!PACKED || 2 * w > (int)blockDim.x) {
        s.nt = blockDim.x;
        s.seg = 0;
        s.lt = threadIdx.x;
        s.nseg = 1;
    } else {
        s.nt = w;
        // segments are whole waves, so the segment (and the row it gives)
        // is wave-uniform: said to the compiler, per-row values (the row's
        // table entries, offsets) load into scalar registers
        s.seg = __builtin_amdgcn_readfirstlane((int)threadIdx.x / w);
        s.lt = (int)threadIdx.x - s.seg * w;
        s.nseg = (int)blockDim.x / w;
    }
    return s;
}

// Deterministic sums of NV values over each segment's threads (the block
// sum when the block holds one row); every thread receives its segment's.
// Segments are whole waves. `red` must hold 16 * NV doubles of LDS.
template <int NV>
__device__ __forceinline__ void seg_sum(double (&v)[NV], double* red, const RowSeg& s) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
    __syncthreads();
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) red[k * 16 + wid] = v[k];
    }
    __syncthreads();
    const int w0 = (s.seg * s.nt) >> 6, nw = (s.nt + 63) >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double t = 0.0;
        for (int w = 0; w < nw; ++w) t += red[k * 16 + w0 + w];
        v[k] = t;
    }
    __syncthreads();
}
// The segment's maximum of a non-negative value.
__device__ __forceinline__ double seg_max(double v, double* red, const RowSeg& s) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    v = wave_max(v);
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    const int w0 = (s.seg * s.nt) >> 6, nw = (s.nt + 63) >> 6;
    double m = 0.0;
    for (int w = 0; w < nw; ++w) m = fmax(m, red[w0 + w]);
    __syncthreads();
    return m;
}
// The line-solve depth of a block's rows: the recorded depth of its one row,
// or the largest over a packed block's rows (every row of a block runs the
// same reduction levels; a deeper reduction than recorded only continues
// an already decoupled one). `red` must hold 16 doubles of LDS.
template <bool PACKED = true>
__device__ __forceinline__ int block_steps(const int* __restrict__ rsteps, int base, int j0,
                                           int nrows, const RowSeg& s, double* red) {
    if (!PACKED || s.nseg == 1) return rsteps[base + j0];
    int mx = -1;
    if (threadIdx.x < 64)
        for (int r = threadIdx.x; r < min(s.nseg, nrows); r += 64) mx = max(mx, rsteps[base + j0 + r]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_xor(mx, o, 64));
    __syncthreads();
    if (threadIdx.x == 0) red[0] = (double)mx;
    __syncthreads();
    const int r = (int)red[0];
    __syncthreads();
    return r;
}

// Sum the per-row partials [base, base+n) of NV interleaved slots
// (layout part[slot * stride + row]).
template <int NV>
__device__ __forceinline__ void sum_partials(const double* __restrict__ part, long stride, int base,
                                             int n, double (&out)[NV], double* red) {
#pragma unroll
    for (int k = 0; k < NV; ++k) out[k] = 0.0;
    for (int r = threadIdx.x; r < n; r += blockDim.x) {
#pragma unroll
        for (int k = 0; k < NV; ++k) out[k] += part[k * stride + base + r];
    }
    block_sum<NV>(out, red);
}

// Per-launch sums of the solve, accumulated without fences: every row block
// adds its block sums with device-scope atomics into one of kAccSub = 64
// sub-accumulators (row j uses j mod 64, so at most nth / 64 atomics meet
// on one address), and kernels of later launches read them (stream order
// makes them visible); a wave reads one slot with one load per lane. Slots
// per bubble: the assembly (|r0|^2, |b|^2, r_in.z, |r_in|^2, mu as a
// maximum) and the FP64 residual of each refinement k = 1..kAccRefine (the
// same first four). A slot is zeroed by a kernel that neither reads nor adds
// to it, before the launch that adds to it: the assembly's by the update
// kernel, refinement 1's by the assembly, refinement k+1's by refinement k.
constexpr int kAccSub = 64, kAccVals = 5, kAccRefine = 16;
constexpr int kAccSlots = 1 + kAccRefine;
constexpr int kAccBubble = kAccSlots * kAccVals * kAccSub;
__host__ __device__ constexpr int acc_slot_res(int k) { return k; }          // k = 0: assembly
__host__ __device__ inline size_t acc_index(int b, int slot, int v, int sub) {
    return (((size_t)b * kAccSlots + slot) * kAccVals + v) * kAccSub + sub;
}
// The sum (maximum) of one value of a slot, in every lane of the calling
// wave; the same in every wave (fixed reduction order).
__device__ __forceinline__ double acc_sum(const double* __restrict__ acc, int b, int slot, int v) {
    return wave_sum(acc[acc_index(b, slot, v, threadIdx.x & 63)]);
}
__device__ __forceinline__ double acc_max(const double* __restrict__ acc, int b, int slot, int v) {
    return wave_max(acc[acc_index(b, slot, v, threadIdx.x & 63)]);
}
__device__ __forceinline__ void acc_add(double* acc, int b, int slot, int v, int sub, double x) {
    unsafeAtomicAdd(acc + acc_index(b, slot, v, sub & (kAccSub - 1)), x);
}
// maximum of non-negative values through their bit patterns
__device__ __forceinline__ void acc_put_max(double* acc, int b, int slot, int v, int sub, double x) {
    atomicMax(reinterpret_cast<unsigned long long*>(acc + acc_index(b, slot, v, sub & (kAccSub - 1))),
              (unsigned long long)__double_as_longlong(x));
}
// zeroes one slot; called by every lane of one wave
__device__ __forceinline__ void acc_zero(double* acc, int b, int slot) {
#pragma unroll
    for (int v = 0; v < kAccVals; ++v) acc[acc_index(b, slot, v, threadIdx.x & 63)] = 0.0;
}

// Flags of SolveCtl that blocks of one launch may set while other blocks of
// the same launch read them: each flag caches a decision every block makes
// from the same sums, so a block sees either value and acts alike.
__device__ __forceinline__ int flag_load(const int* f) {
    return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void flag_store(int* f, int v) {
    __hip_atomic_store(f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The FP64 residual norm the tolerance applies to: relative to |b| unless
// the tolerance is absolute.
__device__ __forceinline__ double residual_norm(double rr, double bb, bool absolute) {
    return absolute ? sqrt(rr) : sqrt(rr) / (bb > 0.0 ? sqrt(bb) : 1.0);
}

// --------------------------------------------- periodic line solve ----
// Reciprocal for the preconditioner: FP32 uses the hardware v_rcp_f32
// (1 ulp; the line solve is a preconditioner, not the residual), FP64 the
// correctly rounded division.
__device__ __forceinline__ float pre_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double pre_rcp(double x) { return 1.0 / x; }

// Coupling below which a reduced row is decoupled: below the rounding of the
// precision, so stopping the reduction there changes z by less than one ulp.
template <typename Ti> struct PcrTol;
template <> struct PcrTol<float> { static constexpr float v = 2e-9f; };
template <> struct PcrTol<double> { static constexpr double v = 1e-18; };

// Parallel cyclic reduction of one periodic tridiagonal row held in LDS,
// normalised to unit diagonal: x_i + a_i x_{i-1} + c_i x_{i+1} = d_i, n a
// power of two >= 4. Each reduction doubles the coupling stride and, for a
// diagonally dominant row, squares the size of the couplings; after
// log2(n)-1 reductions the stride is n/2, where x_{i-n/2} = x_{i+n/2} and
// the rows pair up into 2x2 systems. A row whose couplings have all fallen
// below PcrTol is decoupled early (x_i = d_i).
// steps < 0: reduce adaptively (a block-wide max per reduction) and return
// the number of reductions done; steps >= 0: do exactly that many (the
// count returned by the adaptive solve of the same matrix).
// The reductions alternate between the arrays (sa, sc, sd) and the free
// arrays (ta, tc, td), so one barrier per reduction orders them; on exit
// *x points to the array that holds the solution. CPT bounds the cells per
// thread.
template <typename Ti, int CPT>
__device__ __forceinline__ int pcr_periodic(Ti* sa, Ti* sc, Ti* sd, Ti* ta, Ti* tc, Ti* td, int n,
                                            int steps, float* red, Ti** x, int tid, int nt) {
    const int m = n - 1;
    const int full = 31 - __clz(n) - 1;     // log2(n) - 1
    Ti *a = sa, *c = sc, *d = sd, *na = ta, *nc = tc, *nd = td;
    int done = 0;
    for (int s = 1; s < n / 2; s <<= 1) {
        if (steps >= 0 && done >= steps) break;
        float mx = 0.0f;
#pragma unroll
        for (int k = 0; k < CPT; ++k) {
            int i = tid + k * nt;
            if (i < n) {
                int im = (i - s) & m, ip = (i + s) & m;
                Ti ai = a[i], ci = c[i], di = d[i];
                Ti am = a[im], cm = c[im], dm = d[im];
                Ti ap = a[ip], cp = c[ip], dp = d[ip];
                Ti iD = pre_rcp(Ti(1) - ai * cm - ci * ap);
                const Ti a2 = -ai * am * iD, c2 = -ci * cp * iD;
                na[i] = a2;
                nc[i] = c2;
                nd[i] = (di - ai * dm - ci * dp) * iD;
                mx = fmaxf(mx, (float)(fabs(a2) + fabs(c2)));
            }
        }
        ++done;
        Ti* t;
        t = a; a = na; na = t;
        t = c; c = nc; nc = t;
        t = d; d = nd; nd = t;
        if (steps < 0) {
            // block-wide (every row of a packed block takes the same depth)
            mx = wave_max(mx);
            if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
            __syncthreads();
            float bm = 0.0f;
            for (int w = 0; w < ((int)blockDim.x + 63) >> 6; ++w) bm = fmaxf(bm, red[w]);
            __syncthreads();
            if (bm < (float)PcrTol<Ti>::v) {   // d already holds x
                *x = d;
                return done;
            }
        } else {
            __syncthreads();
        }
    }
    if (done < full) {   // truncated: x_i = d_i
        *x = d;
        return done;
    }
#pragma unroll
    for (int k = 0; k < CPT; ++k) {
        int i = tid + k * nt;
        if (i < n) {
            int j = (i + n / 2) & m;
            Ti ei = a[i] + c[i], ej = a[j] + c[j];
            nd[i] = (d[i] - ei * d[j]) * pre_rcp(Ti(1) - ei * ej);
        }
    }
    __syncthreads();
    *x = nd;
    return done;
}

// The periodic row of a length n that is not a power of two (n >= 2, one
// row per thread: threads t < n hold row t), by the rank-one correction of
// the periodic system into a non-periodic one (Sherman-Morrison; the form of
// Numerical Recipes' `cyclic`): with the corner couplings alpha = a_0 and
// beta = c_{n-1} and gamma = -1, T = T' + u v^T where T' drops the corners
// and has the diagonals 1 - gamma = 2 (row 0) and 1 - alpha beta / gamma =
// 1 + alpha beta (row n-1), u = (gamma, 0, ..., 0, beta), v = (1, 0, ..., 0,
// alpha / gamma). T' y = d and T' z = u are reduced together by
// non-periodic cyclic reduction (a coupling past an end of the row is zero,
// so ceil(log2 n) reductions decouple every row, exactly), and x = y -
// (v . y) / (1 + v . z) z. The arrays (sa, sc, sd, su) and (ta, tc, td, tu)
// alternate as in pcr_periodic; on exit *x points to the solution. Returns
// the number of reductions.
template <typename Ti>
__device__ __forceinline__ int pcr_general(Ti* sa, Ti* sc, Ti* sd, Ti* su, Ti* ta, Ti* tc, Ti* td,
                                           Ti* tu, int n, Ti** x, int i) {
    const bool act = i < n;
    // the corner couplings, read by every thread before rows 0 and n-1 change
    const Ti alpha = sa[0], beta = sc[n - 1];
    __syncthreads();
    if (act) {
        Ti u = Ti(0);
        if (i == 0) {
            sa[0] = Ti(0);
            sc[0] = sc[0] * Ti(0.5);
            sd[0] = sd[0] * Ti(0.5);
            u = Ti(-0.5);
        }
        if (i == n - 1) {
            const Ti inv = Ti(1) / (Ti(1) + alpha * beta);
            sa[i] = sa[i] * inv;
            sc[i] = Ti(0);
            sd[i] = sd[i] * inv;
            u = beta * inv;
        }
        su[i] = u;
    }
    __syncthreads();
    Ti *a = sa, *c = sc, *d = sd, *w = su, *na = ta, *nc = tc, *nd = td, *nw = tu;
    int done = 0;
    for (int s = 1; s < n; s <<= 1) {
        if (act) {
            const int im = i - s, ip = i + s;
            const Ti ai = a[i], ci = c[i];
            Ti am = Ti(0), cm = Ti(0), dm = Ti(0), wm = Ti(0);
            Ti ap = Ti(0), cp = Ti(0), dp = Ti(0), wp = Ti(0);
            if (im >= 0) { am = a[im]; cm = c[im]; dm = d[im]; wm = w[im]; }
            if (ip < n) { ap = a[ip]; cp = c[ip]; dp = d[ip]; wp = w[ip]; }
            const Ti iD = Ti(1) / (Ti(1) - ai * cm - ci * ap);
            na[i] = -ai * am * iD;
            nc[i] = -ci * cp * iD;
            nd[i] = (d[i] - ai * dm - ci * dp) * iD;
            nw[i] = (w[i] - ai * wm - ci * wp) * iD;
        }
        ++done;
        Ti* t;
        t = a; a = na; na = t;
        t = c; c = nc; nc = t;
        t = d; d = nd; nd = t;
        t = w; w = nw; nw = t;
        __syncthreads();
    }
    // d holds y, w holds z
    const Ti f = (d[0] - alpha * d[n - 1]) / (Ti(1) + w[0] - alpha * w[n - 1]);
    if (act) nd[i] = d[i] - f * w[i];
    __syncthreads();
    *x = nd;
    return done;
}

}  // namespace sfk
