// Forward-algorithm kernels for gfx950 (CDNA4, wave64).
//
// The recurrence is the reference's (align_host, gpuworker.cuh:1051-1094;
// GPU kernel pairhmm_kernels.cuh:1417-1763):
//   M[r][c] = lambda(r,c) * (alpha_r M[r-1][c-1] + beta (I[r-1][c-1] + D[r-1][c-1]))
//   I[r][c] = delta_r M[r-1][c] + eps I[r-1][c]
//   D[r][c] = sigma_r M[r][c-1] + eps D[r][c-1]
//   row 0: M = I = 0, D = (FLT_MAX/16)/H;  column 0 (r >= 1): 0
//   score = log10(sum_c M[R][c] + I[R][c]) - log10(FLT_MAX/16)
//
// k_fwd_tile_set -- the hot path.  A wave holds 64/G alignments ("groups") of G
// lanes; lane t of a group holds read rows [t*NR, t*NR+NR) in registers and
// the haplotype streams through the group one column per step (anti-diagonal
// wavefront).  Row-above values cross lanes with DPP wave_shr:1, a group's
// first lane injects the row-0 boundary.  Emission probabilities for the
// 4 bases x NR rows of each lane sit in LDS (one ds_read_b128 per 4 cells,
// conflict-free by lane interleaving; haps holding the wildcard go to
// k_fwd_special).  Its work comes in two units: super-tasks (up to 64/G
// reads of one record against a segment of the record's haps: the wave sets
// the reads up once and sweeps the haps one after another) and items (one
// alignment per group: reads a record leaves over after full chunks, and the
// FP64 rescue lists).  Two arithmetic forms:
//
//  SAFE (6 VALU/cell): variables M, Ib = beta*I, Dh = D/sigma_r.
//    M  = lambda*(alpha M' + Ib' + beta sigma_{r-1} Dh')      fma fma mul
//    Ib = beta delta_r M^ + eps Ib^                            mul fma
//    Dh = M< + eps Dh<                                         fma
//    Magnitudes never exceed the reference's.
//
//  FAST (5 VALU/cell): row-rescaled variables with n_r = prod_{i<=r} alpha_i,
//    Mh = M/n_r, Ih = I/(delta_r n_{r-1}), Dh = D/(sigma_r n_r):
//    Mh = lambda*(Mh' + b_r Ih' + d_r Dh')                     fma fma mul
//    Ih = Mh^ + e_r Ih^                                        fma
//    Dh = Mh< + eps Dh<                                        fma
//    b_r = beta delta_{r-1}/(alpha_{r-1} alpha_r), d_r = beta sigma_{r-1}/alpha_r,
//    e_r = eps delta_{r-1}/(delta_r alpha_{r-1}).  The start constant is
//    lowered by n_R/2 (it cancels in the score) so that every rescaled value
//    stays below FLT_MAX/16; the read pass admits a read only when
//    0 < alpha <= 1, e_r <= 1/2, eps <= 1/2 and n_R >= 1e-30.
//
// Both forms use the reference's out-of-bounds-row trick for the result
// (pairhmm_kernels.cuh:1325-1356): the first row past the read turns the
// I-chain into (M+I) of the last row, later rows pass it through, and the
// lane holding row R accumulates it one column behind.
//
// k_fwd_special -- reads of several tiles and haps with the wildcard.
//
// k_fwd_wave -- one alignment per wave, any read length, FP32 or FP64, with
// the plain (unscaled) recurrence.  Reads longer than the largest tile are
// processed in 64*NR-row tiles whose last row is spilled to global memory
// (the reference's multi-tile kernel, pairhmm_kernels.cuh:2167-3272, keeps a
// border column the same way); the FP64 instance recomputes results whose
// FP32 sum fell below the rescue threshold.
#include "phmm_device.hpp"

namespace phmm {

__device__ __forceinline__ int shr1i(int v)
{
    // DPP wave_shr:1 -- lane i receives lane i-1; lane 0 receives 0 (bound
    // control: an out-of-range source reads as zero).
    return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true);
}
__device__ __forceinline__ float shr1f(float v)
{
    return __int_as_float(shr1i(__float_as_int(v)));
}
__device__ __forceinline__ double shr1d(double v)
{
    const int lo = shr1i(__double2loint(v));
    const int hi = shr1i(__double2hiint(v));
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ int wave_max(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v = max(v, __shfl_xor(v, o, 64));
    return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ int wave_min(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v = min(v, __shfl_xor(v, o, 64));
    return __builtin_amdgcn_readfirstlane(v);
}

// Setup-time division (once per task and row).  FP32: the hardware
// reciprocal times the numerator, within 2 ulp of the quotient.  The
// correctly rounded division is a chain of dependent instructions per row
// that stalls the wave's setup: with it the forward kernel runs about 3%
// slower on 150-base reads against 150-350-base haps.  FP64 (the rescue)
// keeps the correctly rounded quotient.
__device__ __forceinline__ float qdiv(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double qdiv(double a, double b) { return a / b; }

__device__ __forceinline__ float ph2pr_of(const float* table, int q)
{
    return table[q > 127 ? 127 : q];
}

// ---------------------------------------------------------------------------
// k_fwd_tile_set
// ---------------------------------------------------------------------------
template <typename T>
struct TileTraits;
template <>
struct TileTraits<float> {
    typedef float P __attribute__((ext_vector_type(2)));
    // keeps x in an even-aligned register pair -- x.x in an even VGPR, x.y in
    // the odd one above it (no instruction); see tile_sweep's cell
    __device__ static __forceinline__ void pin(P& x) { asm("" : "+v"(x)); }
    using V = float4;  // one ds_read_b128 = 4 rows
    static constexpr int K = 4;
    __device__ static V pack(const float* v) { return make_float4(v[0], v[1], v[2], v[3]); }
    __device__ static void unpack(const V& x, float* v)
    {
        v[0] = x.x;
        v[1] = x.y;
        v[2] = x.z;
        v[3] = x.w;
    }
    __device__ static float shr(float x) { return shr1f(x); }
};
template <>
struct TileTraits<double> {
    typedef double P __attribute__((ext_vector_type(2)));
    __device__ static __forceinline__ void pin(P&) {}
    using V = double2;  // one ds_read_b128 = 2 rows
    static constexpr int K = 2;
    __device__ static V pack(const double* v) { return make_double2(v[0], v[1]); }
    __device__ static void unpack(const V& x, double* v)
    {
        v[0] = x.x;
        v[1] = x.y;
    }
    __device__ static double shr(double x) { return shr1d(x); }
};

// Shape of a lane's emission table in LDS: NV vectors of K rows (the last
// may hold fewer), each for the NL letters (4: the bases; 5: the wildcard of
// the hap too), tab[(q*NL + letter)*64 + lane] --
// one ds_read of 16 bytes per vector, conflict-free because consecutive
// lanes read consecutive 16-byte words; a letter's entry is 64 words on, so
// its address is a shift of the letter whatever NV (a multiply by NV*64
// never issues beside another wave's instruction).  A last vector holding a single row would be
// read as one 4-byte word at a 16-byte lane stride, four lanes to a bank,
// so such a row (kTail) sits in a table of scalars instead,
// stab[letter*64 + lane], at a 4-byte lane stride.
template <typename T, int NR, int NL = 4>
struct TabShape {
    static constexpr int K = TileTraits<T>::K;
    static constexpr bool kTail = K > 1 && NR % K == 1;
    static constexpr int NV = kTail ? NR / K : (NR + K - 1) / K;
    static constexpr int kVecs = NL * NV * 64;
    static constexpr int kWords =  // table size in units of the vector type
        kVecs + (kTail ? (NL * 64 * (int)sizeof(T) + (int)sizeof(typename TileTraits<T>::V) - 1) /
                             (int)sizeof(typename TileTraits<T>::V)
                       : 0);
};

// Per-lane state of a tile task that depends only on the read: its rows'
// coefficients (the emission values of the rows live in the LDS table).
// ROWEPS: every row has its own gap continuation eps_r (per-position gcp
// semantics), so the D chain takes eps_r from a per-row register (FAST: c3;
// SAFE: c4) instead of the lane's eps.
template <typename T, int NR, bool ROWEPS>
struct TileRead {
    typename TileTraits<T>::P c10[NR];  // (c1, c0)
    typename TileTraits<T>::P c32[NR];  // (c3, c2); FAST: b d e eps_r are c0 .. c3, SAFE: alpha w delta' e
    T c4[ROWEPS ? NR : 1];             // SAFE with ROWEPS: eps_r
    T eps, beta;
    int L;
    float nl;
    // log2 of the insertion floor at the lane's last row (the read's last row
    // for the lanes past it), less the start constant's: the product of the
    // rows' chain coefficients, which telescopes -- FAST: eps^R * delta_0 /
    // delta_R / prod(alpha_0 .. alpha_{R-1}); SAFE: eps per row.  The alpha
    // factors (each <= 1) are left out, which can only put the estimate below
    // the true floor.  (In-pass scaling; one gap continuation per read.)
    float floor2;
    double prod;  // strips: product of alpha over the lane's rows
};

// Gap continuation of the D chain of row j.
template <typename T, int NR, bool FAST, bool ROWEPS>
__device__ __forceinline__ T d_eps(const TileRead<T, NR, ROWEPS>& R, int j)
{
    if constexpr (!ROWEPS)
        return R.eps;
    else if constexpr (FAST)
        return R.c32[j].x;
    else
        return R.c4[j];
}

// beta = 1 - eps, rounded as the reference's host code rounds it in FP32
// (float beta = 1.0 - ph2pr[q], gpuworker.cuh:1048).
template <typename T>
__device__ __forceinline__ T beta_of(T e)
{
    if constexpr (sizeof(T) == 4)
        return (T)(float)(1.0 - (double)e);
    else
        return (T)1 - e;
}

// This lane's rows of `read` (inactive lanes: an empty read): coefficients in
// R, emission values in the LDS table.
//
// ROWEPS (per-position gcp): row r (1-based) takes eps_r = ph2pr[gcp[r-1]]
// and beta_r = 1 - eps_r where the reference takes one eps and beta.  FAST:
// b_r = beta_r delta_{r-1}/(alpha_{r-1} alpha_r), d_r = beta_r sigma_{r-1} /
// alpha_r, e_r = eps_r delta_{r-1}/(delta_r alpha_{r-1}), and the D chain
// Dh = Mh< + eps_r Dh<.  SAFE carries Ib_r = beta_{r+1} I_r (the next row's
// beta, so row r+1's M adds it with weight 1): c2 = beta_{r+1} delta_r,
// c3 = eps_r beta_{r+1} / beta_r, and D chain Dh = M< + eps_r Dh<; the last
// row's beta_{L+1} is taken as beta_L, which the epilogue divides out.
//
// row0: the first row of the tile (reads of several tiles).
template <typename T, int NR, bool FAST, bool ROWEPS, int NL = 4>
__device__ __forceinline__ void tile_setup(const FwdParams& p, typename TileTraits<T>::V* tab,
                                           bool active, int read, int t,
                                           TileRead<T, NR, ROWEPS>& R, int row0 = 0)
{
    const BatchDesc& bd = *p.bd;
    using TT = TileTraits<T>;
    constexpr int K = TT::K;
    const int lane = threadIdx.x;
    int L = 0, roff = 0;
    float nl = 1.0f;
    if (active) {
        L = bd.read_len[read];
        roff = bd.read_off[read];
        if (FAST)
            nl = p.meta[read].nl;
    }
    T eps = (T)kEpsGpu, beta = (T)kBetaGpu;
    if (p.semantics != 0 && active && L > 0) {
        // reference CPU semantics: the read's first gcp quality; per-position
        // gcp: the last row's (the SAFE epilogue divides by beta_{L+1} = beta_L)
        const float e = ph2pr_of(p.ph2pr, bd.gcp[roff + (ROWEPS ? L - 1 : 0)]);
        eps = (T)e;
        beta = beta_of((T)e);
    }
    R.eps = eps;
    R.beta = beta;
    R.L = L;
    R.nl = nl;

    // ---- per-row coefficients and the emission table -------------------
    // No branch per row: all of a lane's rows are loaded at once (rows past
    // the read repeat its last one and are selected away), then all their
    // table entries, so that a setup waits twice for memory and not twice per
    // row: 4.56 -> 4.47 ms per call of 10,000 records x 25 reads of 150 bases x
    // 4 haps, with the next hap's loads ahead of a super-task's sweep and the
    // descriptor's pointers in registers.
    const int r0 = row0 + t * NR;
    {
        const int rlast = L > 0 ? L - 1 : 0;
        uint32_t w[NR], wp;
        uint8_t g[ROWEPS ? NR + 1 : 1];
        wp = p.rows[roff + min(max(r0 - 1, 0), rlast)];
#pragma unroll
        for (int j = 0; j < NR; ++j)
            w[j] = p.rows[roff + min(r0 + j, rlast)];
        if constexpr (ROWEPS) {
#pragma unroll
            for (int j = 0; j <= NR; ++j)
                g[j] = bd.gcp[roff + min(r0 + j, rlast)];
        }
        T pb[NR], de[NR], si[NR], er[ROWEPS ? NR + 1 : 1];
#pragma unroll
        for (int j = 0; j < NR; ++j) {  // (row accessors stay within the table)
            pb[j] = (T)p.ph2pr[row_bq(w[j])];
            de[j] = (T)p.ph2pr[row_iq(w[j])];
            si[j] = (T)p.ph2pr[row_dq(w[j])];
        }
        // the row above the lane's first one
        const bool above = r0 >= 1 && r0 - 1 < L;
        T pdelta = above ? (T)p.ph2pr[row_iq(wp)] : (T)0;
        T psigma = above ? (T)p.ph2pr[row_dq(wp)] : (T)0;
        T palpha = above ? (T)1 - (pdelta + psigma) : (T)1;
        if constexpr (ROWEPS) {
#pragma unroll
            for (int j = 0; j <= NR; ++j)
                er[j] = (T)ph2pr_of(p.ph2pr, g[j]);
        }
        // (the clamped loads leave row min(r0 + NR, L) - 1 in w[NR - 1])
        const int lrow = min(r0 + NR, L) - 1;
        R.floor2 = (float)lrow * __log2f((float)eps);
        if (FAST && lrow > 0)
            R.floor2 += __log2f(p.ph2pr[row_iq(p.rows[roff])]) - __log2f((float)de[NR - 1]);
        R.prod = 1.0;
        T lm[NR], lx[NR];
        int code[NR];
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            const int ri = r0 + j;  // 0-based row; 1-based row ri+1
            const bool in = ri < L, top = ri == 0, firstoob = ri == L;
            const T delta = de[j], sigma = si[j];
            const T alpha = (T)1 - (delta + sigma);
            // gap continuation of this row, and (SAFE) the next row's beta
            T e = eps, br = beta, bn = beta;
            if constexpr (ROWEPS) {
                e = er[j];
                br = beta_of(e);
                bn = ri + 1 < L ? beta_of(er[j + 1]) : beta;
            }
            code[j] = in ? row_code(w[j]) : 4;
            lm[j] = in ? (T)1 - pb[j] : (T)0;
            lx[j] = in ? qdiv(pb[j], (T)3) : (T)0;
            if constexpr (NL == 5)
                R.prod *= in ? (double)alpha : 1.0;
            if (FAST) {
                const T c0 = qdiv(br * pdelta, palpha * alpha);
                const T c1 = qdiv(top ? br : br * psigma, alpha);
                const T c2 = qdiv(in ? e * pdelta : pdelta, in ? delta * palpha : palpha);
                R.c10[j].y = in && !top ? c0 : (T)0;
                R.c10[j].x = in ? c1 : (T)0;
                R.c32[j].y = in ? (top ? (T)0 : c2) : firstoob ? c2 : (T)1;
                R.c32[j].x = ROWEPS && in ? e : (T)0;
            } else {
                R.c10[j].y = in ? alpha : (T)0;
                R.c10[j].x = in ? (top ? br : br * psigma) : (T)0;
                R.c32[j].y = in ? bn * delta : firstoob ? beta : (T)0;
                // equal betas keep eps exactly (no rounding of bn / br)
                R.c32[j].x = in ? (bn == br ? e : qdiv(e * bn, br)) : (T)1;
                if constexpr (ROWEPS)
                    R.c4[j] = in ? e : (T)0;
            }
            if (in) {  // rows past the read keep the last row's values
                pdelta = delta;
                psigma = sigma;
                palpha = alpha;
            }
        }
        // emission table: tab[(q*NL + letter)*64 + lane] = rows K*q .. K*q+K-1
        // for the four bases and, with NL 5, a hap's wildcard, which every
        // row matches (a read's 'N' matches every base), a single last row in
        // the scalar table
        using Shape = TabShape<T, NR, NL>;
        constexpr int NV = Shape::NV;
#pragma unroll
        for (int l = 0; l < NL; ++l) {
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                T v[K];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int j = K * q + k;
                    if (j < NR) {
                        const bool m = l == 4 || (l == code[j]) || (code[j] == 4);
                        v[k] = m ? lm[j] : lx[j];
                    } else {
                        v[k] = 0;  // past the lane's rows: never used
                    }
                }
                tab[(q * NL + l) * 64 + lane] = TT::pack(v);
            }
            if constexpr (Shape::kTail) {
                constexpr int j = NR - 1;
                const bool m = l == 4 || (l == code[j]) || (code[j] == 4);
                reinterpret_cast<T*>(tab + Shape::kVecs)[l * 64 + lane] = m ? lm[j] : lx[j];
            }
        }
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            TT::pin(R.c10[j]);
            TT::pin(R.c32[j]);
        }
    }
}

// One cell: row j of the lane's tile at the lane's column, with emission value
// lam.  `up` holds the row above's (M, D) one column back, `chain` its I at
// this column; both move on to this row's.
//
// A SIMD issues a VALU instruction of one wave and, beside it, one of another
// wave -- but beside it only an instruction whose three vector sources do not
// all sit in registers of one parity (measured with two waves: 2.03 cycles
// per FMA with mixed parities, 4.2 with one; a quarter of freely allocated
// FMAs has one).  So M and D of a row are a register pair, M even and D odd,
// and so are its coefficients (c1, c0) and (c3, c2): with chain in M's old
// register every FMA mixes parities.  150-base reads against 150-350-base
// haps: 2.69 -> 2.58 cycles per VALU instruction over the 19-row kernel, 1-2%
// of the call (the clock gives some of it back); over the 16-row kernel, 250-base
// reads against 2-5 kb haps, no gain (0.1% fewer cycles).  The last row's pair is
// only read by the lane transfer, and pinning it cost a move.
template <typename T, int NR, bool FAST, bool ROWEPS>
__device__ __forceinline__ void tile_cell(const TileRead<T, NR, ROWEPS>& R, int j, T lam, T eps,
                                          typename TileTraits<T>::P& md,
                                          typename TileTraits<T>::P& up, T& chain)
{
    const typename TileTraits<T>::P old = md;
    T t1;
    if (FAST) {
        t1 = fma(R.c10[j].x, up.y, up.x);
        t1 = fma(R.c10[j].y, chain, t1);
        chain = fma(R.c32[j].y, chain, up.x);
    } else {
        t1 = fma(R.c10[j].x, up.y, chain);
        t1 = fma(R.c10[j].y, up.x, t1);
        chain = fma(R.c32[j].y, up.x, R.c32[j].x * chain);
    }
    typename TileTraits<T>::P now;
    now.x = lam * t1;
    now.y = fma(eps, old.y, old.x);
    if (j < NR - 1)
        TileTraits<T>::pin(now);
    md = now;
    up = old;
}

// In-pass scaling: the lane above's value of an exponent.  The shifted value
// is kept opaque to the compiler: fused into the subtraction that uses it
// (v_subrev_u32_dpp), it measured as E_{t-1} - E_t on gfx950.
__device__ __forceinline__ int ds_above(int v)
{
    int u = shr1i(v);
    asm volatile("" : "+v"(u));
    return u;
}
// x capped at kDsSpan per lane above the group's lanes over it (x_t <= x_k +
// kDsSpan * (t - k) for k < t: a prefix minimum of x - kDsSpan * t); t: the
// lane's index in its group.
__device__ __forceinline__ int ds_span_cap(int x, int t)
{
    int z = x - kDsSpan * t;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(z, o, 64);
        if (t >= o)
            z = y < z ? y : z;
    }
    return z + kDsSpan * t;
}
// The exponent a lane starts with: its insertion floor (R.floor2) at
// 2^kDsFloor.
__device__ __forceinline__ int ds_start(float C0, float floor2)
{
    const int e0 = (int)floorf((float)kDsFloor - (__log2f(C0) + floor2));
    return e0 < 0 ? 0 : e0;
}
// The exponent of a lane with exponent E that holds or took in values up to
// m (never negative): lowered to put m at 2^kDsGuardTo once it passed
// `guard`, never below 0.
__device__ __forceinline__ int ds_lowered(int E, float m, float guard)
{
    if (!(E > 0 && m > guard))
        return E;
    // v_frexp_exp reads inf as 0: an overflowed lane keeps its exponent and
    // fails acceptance
    const int g = E + kDsGuardTo - (__builtin_amdgcn_frexp_expf(m) - 1);
    return g < 0 ? 0 : g;
}
// The score of a scaled result: the sum a * 2^-E (ok: the sweep's acceptance),
// or, refused, -inf and an entry in `list`.  Returns whether the sum fell
// below the rescue threshold and is finished.
template <bool FAST>
__device__ __forceinline__ bool ds_finish(const FwdParams& p, const WorkItem& it, float a, int E,
                                          bool ok, float nl, float beta, WorkItem* list,
                                          int32_t* count)
{
    if (!ok || !(a >= 0x1p-100f && a <= 3.4028234663852886e38f)) {
        p.bd->scores[it.out] = -INFINITY;
        list[atomicAdd(count, 1)] = it;
        return false;
    }
    // the unscaled sum, where it is a normal float: the score and threshold
    // test of the unscaled instance, bit for bit
    const float at = ldexpf(a, -E);
    float raw;
    if (at >= 0x1p-126f) {
        p.bd->scores[it.out] = FAST ? log10f(at) - (kLog10Scale - kLog10FastKappa)
                                    : log10f(at) - (kLog10Scale + log10f(beta));
        raw = FAST ? at * nl : at / beta;
    } else {
        // a * 2^-E = m * 2^K exactly: the score does not depend on how the
        // rows were split into lanes
        int e2 = 0;
        const float m = frexpf(a, &e2);
        const int K = e2 - E;
        const double off = FAST ? (double)kLog10Scale - (double)kLog10FastKappa
                                : (double)kLog10Scale + log10((double)beta);
        p.bd->scores[it.out] =
            (float)(log10((double)m) + (double)K * 0.30102999566398119521 - off);
        raw = ldexpf(FAST ? a * nl : a / beta, -E);
    }
    return !(raw >= p.rescue_min);
}
// The score of an unscaled FP32 sum; returns whether the sum reached the
// rescue threshold.
template <bool FAST>
__device__ __forceinline__ bool f32_finish(const FwdParams& p, const WorkItem& it, float a, float nl,
                                           float beta)
{
    float score, raw;
    if (FAST) {
        score = log10f(a) - (kLog10Scale - kLog10FastKappa);
        raw = a * nl;
    } else {
        score = log10f(a) - (kLog10Scale + log10f(beta));
        raw = a / beta;
    }
    p.bd->scores[it.out] = score;
    return raw >= p.rescue_min;
}

// One sweep of this group's read (R) against a hap of length HL at hoff;
// the group's result lane writes the score of `it`.  T = float is the first
// pass: results whose FP32 sum (in the reference's units) is below
// rescue_min are appended to the bin's rescue list (rescue_items[rescue_base
// + n], n counted in rescue_counts[bin]).  T = double is the FP64 recompute
// of those lists (start constant 2^1000/H); a result whose sum is not far
// above double's floor goes to the final list.
//
// RE (T = float): the range-extended recompute of the rescue lists.  Lane t
// scales its values by 2^E_t (FwdParams: kReShift and the rule for E_t) --
// the mask multiply that injects the boundary on a group's first lane
// carries the factor 2^(E_t - E_{t-1}) on the others, so the sweep itself is
// unchanged -- and an accepted sum a is exactly a * 2^(kReShift - E_R) of
// the FP32 pass's units.  The magnitude of a lane's last row is read from
// its accumulator: every lane adds up the chain it passes down (only the
// result lane's sum is a score), so a lane above the result lane holds the
// sum over the columns of its last row's outgoing chain -- at no cost in
// the sweep.  The first pass keeps its ilogb for the recompute's scales,
// the recompute checks them with it.
// Returns, for the scaled instances (DS), the number of the wave's
// alignments that fell below the rescue threshold and were finished by the
// scaling (uniform across the wave); 0 otherwise.
// GE: the reference GPU semantics, whose gap continuation is the constant
// kEpsGpu for every read: the D chain's multiplier is then wave-uniform and
// sits in a scalar register, so those FMAs read two vector operands, not
// three (about 1.4% of the sweep's time on gfx950).
// ONE: every group sweeps the same hap (a super-task), so its length needs no
// reduction over the wave.
template <typename T, int NR, bool FAST, bool ROWEPS, bool RE = false, bool DS = false,
          bool GE = false, bool ONE = false>
__device__ __forceinline__ int tile_sweep(const FwdParams& p, const typename TileTraits<T>::V* tab,
                                          const TileRead<T, NR, ROWEPS>& R, bool active, int G,
                                          int t, int HL, int hoff, const WorkItem& it,
                                          int rescue_base, int bin)
{
    const BatchDesc& bd = *p.bd;
    using TT = TileTraits<T>;
    using V = typename TT::V;
    constexpr int K = TT::K;
    constexpr bool F32 = sizeof(T) == 4;
    const int lane = threadIdx.x;
    const bool first = (t == 0);
    const T beta = R.beta;
    const int L = R.L;
    const float nl = R.nl;
    constexpr bool REC = F32 && !ROWEPS && re_rows(NR) && !DS;  // record per-lane magnitudes
    static_assert(!RE || REC, "the range-extended pass is an FP32 pass of the one-eps tiles");
    static_assert(!DS || (F32 && !ROWEPS && !RE && re_rows(NR)),
                  "in-pass scaling: FP32 one-eps tiles of the range-extended rows");
    // the group's lane that forms the sum, the group's first lane and its
    // lanes as a mask (computed where used: nothing extra stays live in
    // the sweep)
    auto res_lane = [&]() { return L / NR; };
    auto group_mask = [&]() {
        return G >= 64 ? ~0ull : (((1ull << G) - 1ull) << (lane - t));
    };

    // ---- wavefront sweep -------------------------------------------------
    typename TT::P MD[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j)
        MD[j] = (T)0;
    T C0 = 0;
    if (active && HL > 0) {
        if (F32)
            C0 = FAST ? (T)((kScale / (float)HL) * (nl * (1.0f / kFastKappa))) : (T)(kScale / (float)HL);
        else
            C0 = FAST ? (T)((kStartF64 / (double)HL) * ((double)nl / (double)kFastKappa))
                      : (T)(kStartF64 / (double)HL);
    }
    // boundary injection: a group's first lane takes row 0 (M = I = 0,
    // D = C0) instead of its left neighbour's last row -- as a multiply by a
    // 0/1 lane mask, which issues at the full FP32 rate where a select does not
    T nf = first ? (T)0 : (T)1;
    int re_E = 0, re_dE = 0;
    bool re_bad = false;
    if constexpr (RE) {
        // per-lane exponents from the FP32 pass's maxima r_k (all lanes of
        // the wave take part in the ballot and shuffles)
        const int slot = active ? it.pad : -1;  // tile_items_task: the rescue-list slot
        const int cm = active && HL > 0 ? ilogbf((float)C0) : 0;
        const int res_t = res_lane(), gbase = lane - t;
        const unsigned long long gmask = group_mask();
        int r = 127;
        if (active && slot >= 0 && t < res_t)
            r = t < kReKnownLanes ? (int)(int8_t)p.rescue_exps[(int64_t)slot * kReKnownLanes + t]
                                  : -128;  // not recorded: extrapolated like an underflow
        re_bad = active && slot < 0;
        const unsigned long long inv = __ballot(active && t < res_t && r < kReValid) & gmask;
        const int lv = (inv ? __ffsll((long long)inv) - 1 - gbase : res_t) - 1;  // last known lane
        const int r_lv = __shfl(r, gbase + (lv > 0 ? lv : 0), 64);
        const int r_lv1 = __shfl(r, gbase + (lv > 1 ? lv - 1 : 0), 64);
        // lanes past the result lane (rows past the read) keep its scale
        const int te = t < res_t ? t : res_t;
        const int r_prev = __shfl(r, gbase + (te > 0 ? te - 1 : 0), 64);
        int E = 0;
        if (te >= 1) {
            if (te - 1 <= lv) {
                E = cm - r_prev;
            } else {
                int slope = lv >= 1 ? r_lv - r_lv1 : lv == 0 ? r_lv - cm : kReUnknownSlope;
                slope = slope < 0 ? slope : 0;
                const int e1 = lv >= 0 ? cm - r_lv : 0;  // E of lane lv + 1
                E = e1 - slope * (te - lv - 1);
            }
        }
        const int Ep = __shfl(E, lane > 0 ? lane - 1 : 0, 64);
        re_dE = t >= 1 ? E - Ep : 0;
        if (active && t <= res_t && (re_dE > 126 || re_dE < -126))
            re_bad = true;
        re_E = E;
        if (!first)
            nf = ldexpf(1.0f, re_dE < -126 ? -126 : re_dE > 126 ? 126 : re_dE);
        C0 = ldexpf((float)C0, -kReShift);
    }
    int ds_E = 0;  // DS: this lane's exponent (held = true * 2^ds_E)
    bool ds_any = false;  // DS: some lane of the wave is scaled (uniform)
    // DS: the transfer factor 2^(E_t - E_{t-1}), exact as long as the
    // exponents stay within kDsSpan
    auto ds_factor = [&]() -> T {
        const int d = ds_E - ds_above(ds_E);
        return first ? (T)0 : (T)ldexpf(1.0f, d);
    };
    if constexpr (DS) {
        // from the floor of the lane's last row (the read's last row for the
        // lanes past it); a group's first lane is not scaled
        int x = 0;
        if (active && C0 > 0 && L > 0 && !first)
            x = ds_start((float)C0, R.floor2);
        if (__ballot(!first && x - ds_above(x) > kDsSpan))  // steep gap scores only
            x = ds_span_cap(x, t);
        ds_E = x;
        nf = ds_factor();
        ds_any = __ballot(ds_E > 0) != 0;
    }
    const T c0f = first ? C0 : (T)0;
    // M and D of the row above reach a lane two steps after they were
    // computed (diagonal dependency), I one step after: step u reads ring
    // entry u % 2 and refills it, so the unrolled steps need no copies
    typename TT::P MDr[2];
    MDr[0].x = MDr[1].x = (T)0;
    MDr[0].y = MDr[1].y = c0f;
    T Iin = 0;
    T acc = 0;

    const int Hmax = ONE ? __builtin_amdgcn_readfirstlane(HL) : wave_max(HL);
    const int nsteps = Hmax + G;
    // Hap letters: lane t consumes column c = s - t at step s.  Each lane
    // keeps a window of two dwords of its hap codes and shifts it by
    // (c mod 4) bytes; dword indices are clamped to the padded hap, so every
    // column up to the padding is exact, and columns outside it (before the
    // lane's first column or past the hap's end) only meet zero state or are
    // never accumulated.
    const uint32_t* hdw = reinterpret_cast<const uint32_t*>(p.hapc + (active ? hoff : 0));
    const int hdw_last = active ? (HL >> 2) : 0;  // padded length / 4 - 1
    const uint32_t shift = (uint32_t)(-t) & 3u;     // (s4 - t) mod 4, constant per lane
    auto hap_dword = [&](int q) { return hdw[min(max(q, 0), hdw_last)]; };
    const int q0 = (0 - t) >> 2;  // floor((s4 - t) / 4) of the first block
    uint32_t wlo = hap_dword(q0), whi = hap_dword(q0 + 1), wnx = hap_dword(q0 + 2);
    // Step s adds the chain of column s - t.  The chain is exactly 0 before
    // a lane's first column, so only the end of the lane's real columns,
    // s <= t + HL, needs a bound: steps below the wave's smallest HL add
    // unconditionally, the rest compare.
    const int acc_last = t + HL;
    const int n_free = (ONE ? Hmax : wave_min(active ? HL : nsteps)) + 1;  // steps s < n_free
    const uint32_t lane_off = lane;  // tab index of this lane's letter-0 entry

    // emission values of step 0; each step loads the next step's values
    // before it computes
    using Shape = TabShape<T, NR>;
    constexpr int NV = Shape::NV;
    const T* stab = reinterpret_cast<const T*>(tab + Shape::kVecs) + lane_off;
    V lam[2][NV];
    T lamS[2] = {(T)0, (T)0};  // the scalar-table row (Shape::kTail)
    uint32_t letters = __builtin_amdgcn_alignbyte(whi, wlo, shift);
    {
        const V* trow = tab + (((letters & 3u) << 6) | lane_off);
#pragma unroll
        for (int qq = 0; qq < NV; ++qq)
            lam[0][qq] = trow[qq * 256];
        if constexpr (Shape::kTail)
            lamS[0] = stab[(letters & 3u) << 6];
    }

    // GE: every lane's eps is kEpsGpu, held in a scalar register (opaque to
    // the compiler, which would otherwise keep the constant in a vector one)
    T eps_ge = (T)0;
    if constexpr (GE) {
        int e = __builtin_bit_cast(int, kEpsGpu);
        asm volatile("" : "+s"(e));
        eps_ge = (T)__builtin_bit_cast(float, e);
    }
    auto sweep4 = [&](int s4, bool bounded) {
        // letters of steps s4+1 .. s4+4: the current window and the next one
        const uint32_t next = __builtin_amdgcn_alignbyte(wnx, whi, shift);
        // The dword after it, a block ahead of its use: loaded at the block's
        // end, the compiler waited for it 50 to 130 instructions later, less
        // than the cache takes (1M reads of 150: 4770 -> 4736 us, 100 records
        // with per-position gcp 8429 -> 8352).  Arithmetic shift: floor.
        const uint32_t wn2 = hap_dword(((s4 - t) >> 2) + 3);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int cur = u & 1, nxt = cur ^ 1;
            // codes are 0..3 inside the hap; the padding's wildcard code
            // reads as base 0 there, and padding columns are never accumulated
            const uint32_t nletter = u < 3 ? (letters >> (8 * (u + 1))) & 3u : next & 3u;
            {
                const V* trow = tab + ((nletter << 6) | lane_off);
#pragma unroll
                for (int qq = 0; qq < NV; ++qq)
                    lam[nxt][qq] = trow[qq * 256];
                if constexpr (Shape::kTail)
                    lamS[nxt] = stab[nletter << 6];
            }
            typename TT::P up = MDr[cur];  // the row above's (M, D), one column back
            T chain = Iin;
            auto cell = [&](int j, T lvk) {
                tile_cell<T, NR, FAST, ROWEPS>(
                    R, j, lvk, GE ? eps_ge : d_eps<T, NR, FAST, ROWEPS>(R, j), MD[j], up, chain);
            };
#pragma unroll
            for (int qq = 0; qq < NV; ++qq) {
                T lv[K];
                TT::unpack(lam[cur][qq], lv);
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int j = K * qq + k;
                    if (j >= (Shape::kTail ? NR - 1 : NR))
                        break;
                    cell(j, lv[k]);
                }
            }
            if constexpr (Shape::kTail)
                cell(NR - 1, lamS[cur]);
            if (bounded)
                acc += (s4 + u <= acc_last) ? chain : (T)0;
            else
                acc += chain;
            // The lane transfers (DPP) never issue beside another wave's
            // instruction, and the older wave of a SIMD goes first in every
            // cycle, so a younger wave stood at each of its transfers until
            // the older one waited for something.  With the priority raised
            // over them they issue at once: 2.89 -> 2.69 cycles per VALU
            // instruction over the 19-row kernel (3-5% of large calls, for
            // two more instructions per step).
            __builtin_amdgcn_s_setprio(3);
            if constexpr (RE) {
                // a group's first lane must not see its neighbour's values:
                // scaled by that alignment's lane factors they may overflow,
                // and inf * 0 would poison this group.  The shifted value is
                // clamped to FLT_MAX first (v_min also maps NaN to it), then
                // masked as in the first pass.  (Not a select: the compiler
                // turns a select of a DPP result into an exec-masked DPP,
                // which reads 0 from the masked-off source lanes.)
                constexpr float kBig = 3.4028234663852886e38f;
                MDr[cur].x = fminf(TT::shr(MD[NR - 1].x), kBig) * nf;
                MDr[cur].y = fma(fminf(TT::shr(MD[NR - 1].y), kBig), nf, c0f);
                Iin = fminf(TT::shr(chain), kBig) * nf;
            } else {
                MDr[cur].x = TT::shr(MD[NR - 1].x) * nf;
                MDr[cur].y = fma(TT::shr(MD[NR - 1].y), nf, c0f);
                Iin = TT::shr(chain) * nf;
            }
            TT::pin(MDr[cur]);
            __builtin_amdgcn_s_setprio(0);
        }
        letters = next;
        wlo = whi;
        whi = wnx;
        wnx = wn2;
    };
    // DS: every kDsEvery steps a scaled lane whose incoming values passed
    // 2^kDsGuard scales down to put them at 2^kDsGuardTo (never below
    // E = 0), rescaling what it holds (the values already taken from the
    // lane above included) and its transfer factor.  Called at wave-uniform
    // points; every lane of the wave takes part in the exchange.
    auto ds_check = [&]() {
        // values are never negative: no absolute values needed
        const float m = fmaxf(fmaxf(fmaxf((float)MDr[0].x, (float)MDr[1].x),
                                    fmaxf((float)MDr[0].y, (float)MDr[1].y)),
                              (float)Iin);
        int x = ds_lowered(ds_E, m, kDsGuardF);
        // any distance in one step: v_ldexp is exact wherever the result
        // stays normal
        if (__ballot(x != ds_E)) {
            // no lane more than kDsSpan above the lane over it, so the
            // transfer factor stays a normal float (a lane whose upper rows
            // meet a read's alignment scales down before its last row, which
            // the lane below sees, does); the scan only where a gap opened
            const int xu = ds_above(x);
            if (__ballot(!first && x - xu > kDsSpan))
                x = ds_span_cap(x, t);
            const int S = x - ds_E;
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                MD[j].x = ldexpf(MD[j].x, S);
                MD[j].y = ldexpf(MD[j].y, S);
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                MDr[k].x = ldexpf(MDr[k].x, S);
                MDr[k].y = ldexpf(MDr[k].y, S);
            }
            Iin = ldexpf(Iin, S);
            acc = ldexpf(acc, S);
            ds_E = x;
            nf = ds_factor();
            ds_any = __ballot(ds_E > 0) != 0;
        }
    };
    int s4 = 0;
    if constexpr (DS) {
        // kDsEvery steps between checks with no branch in between: a
        // branch to the check after every 4 steps cost about 1.3% of the
        // scaled pass (measured on the mixed-length workload)
        static_assert(kDsEvery == 16, "four sweep4 blocks per check");
        for (; s4 + 16 <= n_free && s4 + 12 < nsteps; s4 += 16) {
            sweep4(s4, false);
            sweep4(s4 + 4, false);
            sweep4(s4 + 8, false);
            sweep4(s4 + 12, false);
            if (ds_any)
                ds_check();
        }
    }
    for (; s4 + 4 <= n_free && s4 < nsteps; s4 += 4) {
        sweep4(s4, false);
        if constexpr (DS)
            if (ds_any && (s4 & (kDsEvery - 4)) == kDsEvery - 4)
                ds_check();
    }
    for (; s4 < nsteps; s4 += 4) {
        sweep4(s4, true);
        if constexpr (DS)
            if (ds_any && (s4 & (kDsEvery - 4)) == kDsEvery - 4)
                ds_check();
    }

    if constexpr (RE) {
        // each lane's incoming magnitude, in its own scale: the lane above's
        // chain sum times 2^(E_t - E_{t-1}), within the window
        const float rmp = shr1f((float)acc);
        const int res_t = res_lane();
        bool bad = re_bad;
        if (active && t >= 1 && t <= res_t) {
            if (!(rmp > 0.0f && rmp <= 3.4028234663852886e38f)) {
                bad = true;
            } else {
                const int li = ilogbf(rmp) + re_dE;
                const int cre = ilogbf((float)C0);
                bad = bad || li < cre - kReLow || li > cre + kReHigh;
            }
        }
        const unsigned long long fb = __ballot(bad) & group_mask();
        if (active && t == res_t) {
            const float a = (float)acc;
            if (!fb && a >= 0x1p-100f && a <= 3.4028234663852886e38f) {
                // a * 2^(kReShift - E) = m * 2^K exactly: the score does not
                // depend on how the rows were split into lanes
                int e2 = 0;
                const float m = frexpf(a, &e2);
                const int K = e2 + kReShift - re_E;
                const double off = FAST ? (double)kLog10Scale - (double)kLog10FastKappa
                                        : (double)kLog10Scale + log10((double)(float)beta);
                bd.scores[it.out] =
                    (float)(log10((double)m) + (double)K * 0.30102999566398119521 - off);
            } else {
                const int n = atomicAdd(p.retry_counts + bin, 1);
                p.retry_items[rescue_base + n] = it;
            }
        }
        return 0;
    }
    // DS acceptance: every scaled lane up to the result lane holds a finite
    // running sum (an unscaled lane's sum can overflow harmlessly in the
    // FAST form's upper rows; an overflowed value reaches the result lane's
    // sum), and neighbouring exponents keep the transfer factor a normal
    // float.  Nothing that mattered was flushed: a lane starts with its
    // insertion floor in range and scales down only by what its largest
    // incoming value grew past 2^kDsGuard.
    unsigned long long ds_fb = 0;
    bool ds_done = false;  // finished by the scaling below the rescue threshold
    if constexpr (DS) {
        const int res_t = res_lane();
        const int dl = ds_E - ds_above(ds_E);
        bool bad = false;
        if (active && t <= res_t)
            bad = (ds_E > 0 && !((float)acc <= 3.4028234663852886e38f)) ||
                  (t >= 1 && (dl > 127 || dl < -126));
        ds_fb = __ballot(bad) & group_mask();
    }
    int slot = -1;  // REC: the rescued alignment's rescue-list slot
    if (active && t == L / NR) {
        if (DS && (ds_fb || ds_E > 0 || !((float)acc <= 3.4028234663852886e38f))) {
            ds_done = ds_finish<FAST>(p, it, (float)acc, ds_E, !ds_fb, nl, (float)beta,
                                      p.rescue_items + rescue_base, p.rescue_counts + bin);
        } else if (F32) {
            if (!f32_finish<FAST>(p, it, (float)acc, nl, (float)beta) && p.rescue_on) {
                const int n = atomicAdd(p.rescue_counts + bin, 1);
                p.rescue_items[rescue_base + n] = it;
                if (REC && p.re_on)
                    slot = rescue_base + n;
            }
        } else {
            const double a = (double)acc;
            bd.scores[it.out] = FAST ? (float)(log10(a) - (kLog10StartF64 - log10((double)kFastKappa)))
                                     : (float)(log10(a) - log10((double)beta) - kLog10StartF64);
            // one scale for the whole alignment: accept sums that stay far
            // above double's floor (score above ~ -572), where no cell that
            // matters can have been flushed; the rest go to the
            // exponent-tracking wave kernel
            if (!(a >= 0x1p-900 && a < 1e300)) {
                const int n = atomicAdd(p.final_count, 1);
                p.final_items[n] = it;
            }
        }
    }
    if constexpr (REC) {
        // the group's lanes above the result lane store their magnitudes for
        // the range-extended pass
        const int res_t = res_lane();
        const int gs = __shfl(slot, lane - t + (res_t < G ? res_t : G - 1), 64);
        if (gs >= 0 && active && t < res_t && t < kReKnownLanes) {
            const int e = acc > 0.0f ? ilogbf((float)acc) : -128;
            p.rescue_exps[(int64_t)gs * kReKnownLanes + t] =
                (uint8_t)(int8_t)(e < -128 ? -128 : e > 127 ? 127 : e);
        }
    }
    if constexpr (DS)
        return __popcll(__ballot(ds_done));
    return 0;
}

// A task of 64/G consecutive alignments of an item list (the FP64 recompute
// of rescue lists): every group sets up its own read and sweeps its own hap.
template <typename T, int NR, bool FAST, bool ROWEPS, bool RE = false, bool DS = false,
          bool GE = false>
__device__ __forceinline__ int tile_items_task(const FwdParams& p, typename TileTraits<T>::V* tab,
                                                const WorkItem* items, int begin, int count, int G,
                                                int task, int rescue_base, int bin)
{
    const BatchDesc& bd = *p.bd;
    const int lane = threadIdx.x;
    const int W = 64 / G;
    const int grp = lane / G;
    const int t = lane - grp * G;
    const int local = task * W + grp;
    const bool active = grp < W && local < count;
    WorkItem it;
    it.read = 0;
    it.hap = 0;
    it.out = -1;
    it.pad = 0;
    if (active) {
        it = items[begin + local];
        if (RE)
            it.pad = begin + local;  // the rescue-list slot: its maxima in rescue_exps
    }
    TileRead<T, NR, ROWEPS> R;
    tile_setup<T, NR, FAST, ROWEPS>(p, tab, active, it.read, t, R);
    const int HL = active ? bd.hap_len[it.hap] : 0;
    const int hoff = active ? bd.hap_off[it.hap] : 0;
    return tile_sweep<T, NR, FAST, ROWEPS, RE, DS, GE>(p, tab, R, active, G, t, HL, hoff, it,
                                                       rescue_base, bin);
}

// A super-task: the groups set up their reads once and sweep the segment's
// haps in turn (all groups share each hap, so every sweep is uniform across
// the wave).  Empty haps were scored -inf by the scatter; haps holding a
// byte other than A/C/G/T have bins of their own.
template <typename T, int NR, bool FAST, bool ROWEPS, bool DS = false, bool GE = false>
__device__ __forceinline__ int tile_super_task(const FwdParams& p, typename TileTraits<T>::V* tab,
                                               const SuperTask& st, int G, int rescue_base, int bin)
{
    const BatchDesc& bd = *p.bd;
    const int lane = threadIdx.x;
    const int W = 64 / G;
    const int grp = lane / G;
    const int t = lane - grp * G;
    const bool active = grp < W && grp < (st.nc & 0xff);
    const int rd = active ? p.read_perm[st.perm + grp] : 0;
    TileRead<T, NR, ROWEPS> R;
    tile_setup<T, NR, FAST, ROWEPS>(p, tab, active, rd, t, R);
    int done = 0;
    // the next hap's length, offset and flag are loaded before a sweep
    int hl_next = bd.hap_len[st.h0 + st.hs], off_next = bd.hap_off[st.h0 + st.hs];
    int flag_next = p.hapflag[st.h0 + st.hs];
    for (int h = st.hs; h < st.he; ++h) {
        const int hap = st.h0 + h;
        const int HL = hl_next, hoff = off_next, flag = flag_next;
        if (h + 1 < st.he) {
            hl_next = bd.hap_len[hap + 1];
            off_next = bd.hap_off[hap + 1];
            flag_next = p.hapflag[hap + 1];
        }
        if (HL <= 0 || flag != 0)
            continue;
        WorkItem it;
        it.read = rd;
        it.hap = hap;
        it.out = st.aoff + (rd - st.r0) * st.nh + h;
        it.pad = 0;
        done += tile_sweep<T, NR, FAST, ROWEPS, false, DS, GE, true>(p, tab, R, active, G, t, HL, hoff, it,
                                                              rescue_base, bin);
    }
    return done;
}

// Lane i < bs.n of a wave describes bin i of a BinSet: its id, lanes per
// alignment, begin, count and number of tasks (`per_task` units per task;
// 0: one super-task per task in super-task bins, 64 / lanes items per task
// in the others); incl is the inclusive prefix of tasks over the lanes.
// Returns the total number of tasks.
struct SetLane {
    int bin, G, begin, count, ntask, incl;
};
__device__ __forceinline__ int set_lanes(const BinSet& bs, int per_task, SetLane& s)
{
    const int lane = threadIdx.x;
    s.bin = 0;
    s.G = 1;
    s.begin = 0;
    s.count = 0;
    s.ntask = 0;
    if (lane < bs.n) {
        s.bin = bs.bin[lane];
        s.G = bs.lanes[lane] > 0 ? bs.lanes[lane] : 1;
        s.count = bs.counts[(int64_t)bs.count_stride * s.bin];
        s.begin = bs.range ? bs.range[2 * s.bin] : 0;
        const int per = per_task > 0                            ? per_task
                        : (bs.st && s.bin < bs.item_bin0) ? 1
                                                          : 64 / s.G;
        s.ntask = (s.count + per - 1) / per;
    }
    int x = s.ntask;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o)
            x += y;
    }
    s.incl = x;
    return __shfl(x, 63, 64);
}

// The lane (bin) whose task range holds `task` (task < total).
__device__ __forceinline__ int set_find(const SetLane& s, int task)
{
    const unsigned long long m = __ballot(s.incl > task);
    return __ffsll((long long)m) - 1;
}

// Tasks of a persistent launch.  2048 waves that all take their first task
// from the launch's counter stand in line for it: the last one starts 20 us
// after the first.  So with few tasks per block, block b starts on task b and
// only later tasks come from the counter, and a launch of no more tasks than
// blocks touches none: 250 reads against 32 haps 244.9 -> 226.4 us, 1000
// records of 8 x 4 316.6 -> 299.6 us.  With many, the blocks start on the last
// tasks instead and then take the others from the first on: tasks come largest
// first, and a block that becomes resident late, behind another launch's
// blocks, then holds back a small one (1000 records of up to 500 reads of 30 to
// 250 bases: 42970 us all from the counter, 43814 from the front, 42357 from
// the end).  In between neither holds: from the end, large tasks start too late
// (400 records of 16 x 8 with 2-5 kb haps: 5417 us, 5312 from the counter), and
// from the front they are held back (300 records of the mixed batch: 13290 us,
// 13100 from the counter).  `blocks`: the blocks that take tasks, the first
// ones of the launch.
__device__ __forceinline__ int counter_task(int32_t* ctr)
{
    int t = 0;
    if (threadIdx.x == 0)
        t = atomicAdd(ctr, 1);
    return __shfl(t, 0, 64);
}
constexpr int kFrontRounds = 4, kTailRounds = 8;  // tasks per block
__device__ __forceinline__ int next_task(int32_t* ctr, int total, int blocks, bool first)
{
    const bool front = total < kFrontRounds * blocks, tail = total >= kTailRounds * blocks;
    if (first && (front || tail))
        return tail ? total - 1 - (int)blockIdx.x : (int)blockIdx.x;
    if (total <= blocks)
        return total;
    const int t = counter_task(ctr) + (front ? blocks : 0);
    return tail && t >= total - blocks ? total : t;
}

// Waves per SIMD a tile kernel is built for: the 12-row tiles and the
// 13-row FAST tile fit three (at most 168 VGPRs, no spills) and issue more
// of their dependent FMA chains per cycle that way; the larger tiles need
// up to 256 VGPRs and run two.
// The range-extended instances (a smaller share of the time, and a few more
// live values in setup) are not held to three.
// The scaled instances are held to two where the register file allows no
// more (the 20-row SAFE tile would otherwise take AGPRs and run one).
template <typename T, int NR, bool FAST, bool RE, bool DS>
constexpr int tile_waves_per_simd()
{
    return (sizeof(T) == 4 && !RE && (NR == 12 || (NR == 13 && FAST))) ? 3 : DS ? 2 : 1;
}

// Bins of one template in one persistent launch: each wave takes a task, then
// the next one (next_task).  Consecutive tasks of a length-sorted bin have
// similar lengths, and a wave that finishes early takes the next one.  Returns
// the alignments the scaling finished below the threshold (DS).
template <typename T, int NR, bool FAST, bool ROWEPS, bool RE, bool DS, bool GE>
__device__ __forceinline__ int tile_set_tasks(const FwdParams& p, const BinSet& bs,
                                              typename TileTraits<T>::V* tab, const SetLane& sl,
                                              int total)
{
    int done = 0;
    for (int task = next_task(bs.next_task, total, gridDim.x, true); task < total;
         task = next_task(bs.next_task, total, gridDim.x, false)) {
        // the task's bin, in scalar registers (uniform across the wave)
        const int k = set_find(sl, task);
        const int bin = __builtin_amdgcn_readfirstlane(__shfl(sl.bin, k, 64));
        const int G = __builtin_amdgcn_readfirstlane(__shfl(sl.G, k, 64));
        const int begin = __builtin_amdgcn_readfirstlane(__shfl(sl.begin, k, 64));
        const int count = __builtin_amdgcn_readfirstlane(__shfl(sl.count, k, 64));
        const int t0 = __builtin_amdgcn_readfirstlane(__shfl(sl.incl - sl.ntask, k, 64));
        // an item bin's results below the threshold join its tile bin's list
        const int rbin = bin >= bs.item_bin0 ? bin - bs.item_bin0 : bin;
        const int rescue_base =
            __builtin_amdgcn_readfirstlane(bs.seg ? bs.seg[2 * rbin] : 0);
        if constexpr (!RE) {
            if (bs.st && bin < bs.item_bin0) {
                done += tile_super_task<T, NR, FAST, ROWEPS, DS, GE>(
                    p, tab, bs.st[begin + (task - t0)], G, rescue_base, rbin);
                continue;
            }
        }
        done += tile_items_task<T, NR, FAST, ROWEPS, RE, DS, GE>(p, tab, bs.items, begin, count,
                                                                 G, task - t0, rescue_base, rbin);
    }
    return done;
}

template <typename T, int NR, bool FAST, bool ROWEPS = false, bool RE = false, bool DS = false>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(tile_waves_per_simd<T, NR, FAST, RE, DS>(), 8))) void k_fwd_tile_set(
    FwdParams p, BinSet bs)
{
    static_assert(NR >= 4 && NR <= 32, "rows per lane");
    __shared__ typename TileTraits<T>::V tab[TabShape<T, NR>::kWords];
    SetLane sl;
    const int total = set_lanes(bs, 0, sl);
    if (total == 0)  // empty bins (common in a persistent launch): no atomic traffic
        return;
    // the descriptor's pointers in registers: behind p.bd every use of one in
    // a task would wait for the pointer first
    const BatchDesc bd = *p.bd;
    p.bd = &bd;
    // DS: alignments finished by the scaling below the threshold.  The
    // scaled instances (the default FP32 pass) carry a copy of the sweep
    // for the reference GPU semantics, whose eps is one constant.
    int done;
    if (DS && !ROWEPS && p.semantics == 0)
        done = tile_set_tasks<T, NR, FAST, ROWEPS, RE, DS, DS && !ROWEPS>(p, bs, tab, sl, total);
    else
        done = tile_set_tasks<T, NR, FAST, ROWEPS, RE, DS, false>(p, bs, tab, sl, total);
    if constexpr (DS)
        if (done > 0 && threadIdx.x == 0)
            atomicAdd(p.scaled_total, (unsigned long long)done);
}

// ---------------------------------------------------------------------------
// k_fwd_wave
// ---------------------------------------------------------------------------
template <typename T>
struct WaveScalar;
template <>
struct WaveScalar<float> {
    __device__ static float shr(float v) { return shr1f(v); }
    __device__ static float ldexp(float v, int k) { return ldexpf(v, k); }
    __device__ static int ilogb(float v) { return ilogbf(v); }
    // ilogb of a positive finite value in one instruction
    __device__ static int expo(float v) { return __builtin_amdgcn_frexp_expf(v) - 1; }
};
template <>
struct WaveScalar<double> {
    __device__ static double shr(double v) { return shr1d(v); }
    __device__ static double ldexp(double v, int k) { return ::ldexp(v, k); }
    __device__ static int ilogb(double v) { return ::ilogb(v); }
    __device__ static int expo(double v) { return __builtin_amdgcn_frexp_exp(v) - 1; }
};

// k_fwd_wave's arithmetic for reads of one tile, `take` items (reads below 64 *
// NR bases, no byte that matches nothing but itself, one gap continuation per
// read) side by side on the wave, G lanes each.  What differs is how the
// emission values are found: in an LDS table of five letters (as
// tile_setup's), with the letters loaded four columns ahead, where k_fwd_wave
// compares codes.
template <typename T, int NR>
__device__ __forceinline__ void pack_task(const FwdParams& p, typename TileTraits<T>::V* tab,
                                          const WorkItem* items, int take, int G)
{
    using S = WaveScalar<T>;
    using V = typename TileTraits<T>::V;
    constexpr int K = TileTraits<T>::K, NV = NR / K, NL = 5;
    static_assert(NR % K == 0, "whole vectors");
    constexpr int kNone = -(1 << 28);
    const BatchDesc& bd = *p.bd;
    const int lane = threadIdx.x, grp = lane / G, t = lane - grp * G;
    const bool active = grp < take;
    WorkItem it;
    it.read = 0;
    it.hap = 0;
    it.out = -1;
    it.pad = 0;
    if (active)
        it = items[grp];
    const int L = active ? bd.read_len[it.read] : 0, HL = active ? bd.hap_len[it.hap] : 0;
    const int roff = active ? bd.read_off[it.read] : 0;
    T eps = (T)kEpsGpu, beta = (T)kBetaGpu;
    if (p.semantics == 1 && active) {
        const float e = ph2pr_of(p.ph2pr, bd.gcp[roff]);
        eps = (T)e;
        beta = (T)1 - (T)e;
    }
    const T C0 = active ? S::ldexp((T)1, 64) / (T)HL : (T)0;
    T ca[NR], cb[NR], cdl[NR], cs[NR], ce[NR];
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        T lm[K], lx[K];
        int code[K];
#pragma unroll
        for (int x = 0; x < K; ++x) {
            const int j = K * q + x, ri = t * NR + j;
            if (ri < L) {
                const uint32_t w = p.rows[roff + ri];
                const T pb = (T)ph2pr_of(p.ph2pr, row_bq(w));
                const T de = (T)ph2pr_of(p.ph2pr, row_iq(w));
                const T si = (T)ph2pr_of(p.ph2pr, row_dq(w));
                ca[j] = (T)1 - (de + si);
                cb[j] = beta;
                cdl[j] = de;
                cs[j] = si;
                ce[j] = eps;
                lm[x] = (T)1 - pb;
                code[x] = row_code(w);
                lx[x] = code[x] == 4 ? lm[x] : pb / (T)3;
            } else {
                ca[j] = 0;
                cb[j] = 0;
                cdl[j] = ri == L ? (T)1 : (T)0;
                cs[j] = 0;
                ce[j] = 1;
                lm[x] = 0;
                lx[x] = 0;
                code[x] = 4;
            }
        }
#pragma unroll
        for (int l = 0; l < NL; ++l) {
            T v[K];
#pragma unroll
            for (int x = 0; x < K; ++x)
                v[x] = l == 4 || l == code[x] ? lm[x] : lx[x];
            tab[(q * NL + l) * 64 + lane] = TileTraits<T>::pack(v);
        }
    }
    T M[NR], D[NR];
#pragma unroll
    for (int j = 0; j < NR; ++j) {
        M[j] = 0;
        D[j] = 0;
    }
    int sc = 0, sc_end = 0;
    T acc = 0, acc_end = 0, C0s = C0;
    T Ml = 0, Dl = t == 0 ? C0 : (T)0, Mul = 0, Dul = Dl, Iin = 0;
    const int tr = L / NR;
    auto rescale = [&](int kk) {
#pragma unroll
        for (int j = 0; j < NR; ++j) {
            M[j] = S::ldexp(M[j], kk);
            D[j] = S::ldexp(D[j], kk);
        }
        Ml = S::ldexp(Ml, kk);
        Dl = S::ldexp(Dl, kk);
        Mul = S::ldexp(Mul, kk);
        Dul = S::ldexp(Dul, kk);
        Iin = S::ldexp(Iin, kk);
        acc = S::ldexp(acc, kk);
        C0s = S::ldexp(C0s, kk);
        sc -= kk;
    };
    auto fit = [&](int e_in) {
        T my = fmax(fmax(fmax(Ml, Dl), fmax(Mul, Dul)), fmax(Iin, acc));
#pragma unroll
        for (int j = 0; j < NR; ++j)
            my = fmax(my, fmax(M[j], D[j]));
        const int e_my = my > (T)0 ? S::expo(my) : kNone;
        const int e = e_in > e_my ? e_in : e_my;
        if (e > kNone && (e > 96 || e < -32))
            rescale(64 - e);
    };
    auto expo = [&](T v, int e) { return v > (T)0 ? S::expo(v) + e : kNone; };
    // the letters of four columns at a time, the next four loaded ahead;
    // columns outside the hap read as the wildcard
    const uint32_t* hdw = reinterpret_cast<const uint32_t*>(p.hapc + (active ? bd.hap_off[it.hap] : 0));
    const int hdw_last = HL >> 2;
    const uint32_t shift = (uint32_t)(-t) & 3u;
    auto hap_dword = [&](int q) { return hdw[min(max(q, 0), hdw_last)]; };
    const int q0 = (0 - t) >> 2;
    uint32_t wlo = hap_dword(q0), whi = hap_dword(q0 + 1), wnx = hap_dword(q0 + 2);
    auto emission = [&](int c, uint32_t code, V (&lam)[NV]) {
        const uint32_t letter = (uint32_t)c < (uint32_t)HL ? code & 7u : 4u;
        const V* trow = tab + ((letter << 6) | lane);
#pragma unroll
        for (int q = 0; q < NV; ++q)
            lam[q] = trow[q * (NL * 64)];
    };
    const int nsteps = wave_max(active ? HL + tr + 1 : 0);
    V lam[2][NV];
    uint32_t letters = __builtin_amdgcn_alignbyte(whi, wlo, shift);
    emission(-t, letters, lam[0]);
    for (int s4 = 0; s4 < nsteps; s4 += 4) {
        const uint32_t next = __builtin_amdgcn_alignbyte(wnx, whi, shift);
        wlo = whi;
        whi = wnx;
        wnx = hap_dword(((s4 - t) >> 2) + 3);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int s = s4 + u, c = s - t;
            emission(c + 1, u < 3 ? letters >> (8 * (u + 1)) : next, lam[(u + 1) & 1]);
            T mp = Mul, dp = Dul, chain = Iin;
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                T lv[K];
                TileTraits<T>::unpack(lam[u & 1][q], lv);
#pragma unroll
                for (int x = 0; x < K; ++x) {
                    const int j = K * q + x;
                    const T mo = M[j], dov = D[j];
                    M[j] = lv[x] * (ca[j] * mp + cb[j] * (chain + dp));
                    chain = cdl[j] * mp + ce[j] * chain;
                    D[j] = cs[j] * mo + ce[j] * dov;
                    mp = mo;
                    dp = dov;
                }
            }
            if (t == tr && c >= 1 && c <= HL)
                acc += chain;
            if (c == HL) {  // the sum is complete: see k_fwd_wave
                acc_end = acc;
                sc_end = sc;
            }
            const T sM = S::shr(M[NR - 1]), sD = S::shr(D[NR - 1]), sI = S::shr(chain);
            const int ssc = shr1i(sc);
            int e_in = kNone;
            if (t != 0) {
                e_in = expo(sM, ssc - sc);
                const int e2 = expo(sD, ssc - sc), e3 = expo(sI, ssc - sc);
                e_in = e2 > e_in ? e2 : e_in;
                e_in = e3 > e_in ? e3 : e_in;
            }
            fit(e_in);
            const int d = ssc - sc;
            Mul = Ml;
            Dul = Dl;
            Ml = t == 0 ? (T)0 : S::ldexp(sM, d);
            Dl = t == 0 ? C0s : S::ldexp(sD, d);
            Iin = t == 0 ? (T)0 : S::ldexp(sI, d);
        }
        letters = next;
    }
    if (active && t == tr) {
        const double lg = log10((double)acc_end) + (double)sc_end * 0.30102999566398119521 -
                          log10((double)C0 * (double)HL);
        bd.scores[it.out] = (float)lg;
        const double lmin = log10((double)p.rescue_min) - (double)kLog10Scale;
        if (sizeof(T) == 4 && p.rescue_on && !(acc_end > (T)0 && lg >= lmin && lg < 1e30))
            p.final_items[atomicAdd(p.final_count, 1)] = it;
    }
}

// The items are those of the BinSet, one wave each (blocks take every
// gridDim-th item of the bins' concatenated item sequence).  `spill` holds
// spill_elems values of T; each resident block holds the border row's M, I,
// D per column and the power-of-two exponents they were stored with.
//
// Values carry a per-lane power-of-two exponent `sc` (true = stored * 2^sc).
// Before a lane takes in values from the lane above (or, for lane 0 of a
// lower tile, from the spilled border row) it compares their exponent, in
// its own scale, with its own largest value and rescales itself when the
// larger of the two leaves [2^-32, 2^96]; so nothing it receives can
// overflow or vanish, and the result is finite however low the score.  The sum
// is taken at the hap's last column: past it every letter matches, so that the
// values of a read hanging over the hap grow, and with the sum scaled down
// beside them its bits were flushed (scores between -75 and -65 off by up to
// 0.24).
// T = float (multi-tile first pass) appends results below the rescue
// threshold (as the tile kernels define it) to the final list, which the
// T = double instance recomputes.
// PACK: runs of items that pack_task takes go to it instead.
template <typename T, int NR, bool PACK = false>
__global__ __launch_bounds__(64) void k_fwd_wave(FwdParams p, BinSet bs, const int32_t* hmax_ptr,
                                                 T* spill, int64_t spill_elems,
                                                 int32_t* error_flag, int64_t* totals)
{
    using S = WaveScalar<T>;
    const BatchDesc& bd = *p.bd;
    constexpr int TR = 64 * NR;
    constexpr int kNone = -(1 << 28);
    const int lane = threadIdx.x;
    SetLane sl;
    const int n = set_lanes(bs, 1, sl);  // one item per wave
    const int n0 = __shfl(sl.ntask, 0, 64);
    if (totals && blockIdx.x == 0 && lane < 2 && n0 > 0)
        atomicAdd(reinterpret_cast<unsigned long long*>(totals + lane), (unsigned long long)n0);
    const int hmax = *hmax_ptr;
    // per block: 3*(hmax+1) values of T, then 2*(hmax+1) int32 exponents,
    // in units of T (rounded up to 16 bytes)
    const int64_t bytes = 3 * (int64_t)(hmax + 1) * (int64_t)sizeof(T) + 8 * (int64_t)(hmax + 1);
    const int64_t stride = ((bytes + 15) / 16) * 16 / (int64_t)sizeof(T);
    const int64_t cap_blocks = spill_elems / stride;
    const int nblk = (int)(cap_blocks < (int64_t)gridDim.x ? cap_blocks : (int64_t)gridDim.x);
    if (nblk <= 0) {
        if (blockIdx.x == 0 && lane == 0 && n > 0)
            *(volatile int32_t*)error_flag = 1;
        return;
    }
    if ((int)blockIdx.x >= nblk)
        return;
    T* sp = spill + (int64_t)blockIdx.x * stride;
    // per column c: sp[3c+0] = M, sp[3c+1] = I, sp[3c+2] = D of the border
    // row; ex[2c] / ex[2c+1] the exponents M/D and I were stored with
    int32_t* ex = reinterpret_cast<int32_t*>(sp + 3 * (int64_t)(hmax + 1));

    // PACK: runs of three items (as many as fit side by side for reads of up
    // to 167 bases at 8 rows per lane), shorter where the blocks outnumber them
    const int run = PACK ? max(1, min(3, (n + nblk - 1) / nblk)) : 1;
    for (int v = blockIdx.x * run; v < n; v += nblk * run)
    for (int w = v; w < min(n, v + run); ++w) {
        if constexpr (PACK) {
            __shared__ typename TileTraits<T>::V tab[5 * (NR / TileTraits<T>::K) * 64];
            const int kq = set_find(sl, w);
            const int wq = __shfl(sl.incl - sl.ntask, kq, 64);
            const WorkItem* q = bs.items + __shfl(sl.begin, kq, 64) + (w - wq);
            const int rem = min(__shfl(sl.incl, kq, 64), v + run) - w;  // within the bin
            int L = 0;
            bool ok = true;
            if (lane < rem) {
                const int hl = bd.hap_len[q[lane].hap];
                L = bd.read_len[q[lane].read];
                ok = p.semantics == 0 && L > 0 && L < TR && hl > 0 && hl <= hmax;
            }
            if (!__ballot(!ok)) {
                const int G = (wave_max(L) + NR) / NR;  // ceil((L + 1) / NR)
                const int take = min(rem, 64 / G);
                pack_task<T, NR>(p, tab, q, take, G);
                w += take - 1;
                continue;
            }
        }
        const int kb = set_find(sl, w);
        const int begin = __shfl(sl.begin, kb, 64);
        const int w0 = __shfl(sl.incl - sl.ntask, kb, 64);
        const WorkItem it = bs.items[begin + (w - w0)];
        const int L = bd.read_len[it.read];
        const int HL = bd.hap_len[it.hap];
        const int roff = bd.read_off[it.read];
        const int hoff = bd.hap_off[it.hap];
        if (L <= 0 || HL <= 0) {
            if (lane == 0)
                bd.scores[it.out] = -INFINITY;
            continue;
        }
        if (HL > hmax) {
            if (lane == 0) {
                *(volatile int32_t*)(error_flag + 1) = 1;
                bd.scores[it.out] = __int_as_float(0x7fc00000);
            }
            continue;
        }
        // gap continuation: fixed (reference GPU semantics), the read's first
        // gcp quality (reference CPU semantics) or every row's own
        // (per-position gcp, set per row below)
        T eps = (T)kEpsGpu, beta = (T)kBetaGpu;
        if (p.semantics == 1) {
            const float e = ph2pr_of(p.ph2pr, bd.gcp[roff]);
            eps = (T)e;
            beta = (T)1 - (T)e;
        }
        const bool row_gcp = p.semantics == 2;
        const T C0 = S::ldexp((T)1, 64) / (T)HL;
        const int ntiles = (L + 1 + TR - 1) / TR;
        // Emission match: codes with 4 as the wildcard (reference GPU
        // semantics), or the raw bytes with a literal 'N' as the wildcard
        // (reference CPU semantics, gpuworker.cuh:1063) -- exact for any byte.
        const bool raw = p.semantics != 0;
        const int wild = raw ? (int)'N' : 4;
        T acc = 0, acc_end = 0;
        int sc = 0, sc_end = 0;
        for (int k = 0; k < ntiles; ++k) {
            const int r0 = k * TR + lane * NR;
            T ca[NR], cb[NR], cdl[NR], cs[NR], ce[NR], lm[NR], lx[NR];
            int code[NR];
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int ri = r0 + j;
                if (ri < L) {
                    const uint32_t w32 = p.rows[roff + ri];
                    const T pb = (T)ph2pr_of(p.ph2pr, row_bq(w32));
                    const T de = (T)ph2pr_of(p.ph2pr, row_iq(w32));
                    const T si = (T)ph2pr_of(p.ph2pr, row_dq(w32));
                    ca[j] = (T)1 - (de + si);
                    cdl[j] = de;
                    cs[j] = si;
                    if (row_gcp) {
                        const T e = (T)ph2pr_of(p.ph2pr, bd.gcp[roff + ri]);
                        ce[j] = e;
                        cb[j] = (T)1 - e;
                    } else {
                        ce[j] = eps;
                        cb[j] = beta;
                    }
                    lm[j] = (T)1 - pb;
                    code[j] = raw ? (int)bd.read_data[roff + ri] : row_code(w32);
                    lx[j] = code[j] == wild ? lm[j] : pb / (T)3;
                } else {
                    ca[j] = 0;
                    cb[j] = 0;
                    cdl[j] = ri == L ? (T)1 : (T)0;
                    cs[j] = 0;
                    ce[j] = 1;
                    lm[j] = 0;
                    lx[j] = 0;
                    code[j] = wild;
                }
            }
            T M[NR], D[NR];
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                M[j] = 0;
                D[j] = 0;
            }
            const bool top = (k == 0);
            sc = 0;
            acc = 0;
            T C0s = C0;
            T Ml = 0, Dl = (lane == 0 && top) ? C0 : (T)0, Mul = 0, Dul = Dl, Iin = 0;
            const bool last_tile = (k == ntiles - 1);
            const int tr = last_tile ? (L - k * TR) / NR : -1;
            const int nsteps = HL + (last_tile ? tr : 63) + 1;
            auto rescale = [&](int kk) {
#pragma unroll
                for (int j = 0; j < NR; ++j) {
                    M[j] = S::ldexp(M[j], kk);
                    D[j] = S::ldexp(D[j], kk);
                }
                Ml = S::ldexp(Ml, kk);
                Dl = S::ldexp(Dl, kk);
                Mul = S::ldexp(Mul, kk);
                Dul = S::ldexp(Dul, kk);
                Iin = S::ldexp(Iin, kk);
                acc = S::ldexp(acc, kk);
                C0s = S::ldexp(C0s, kk);
                sc -= kk;
            };
            // make room for incoming values of exponent e_in (own scale)
            auto fit = [&](int e_in) {
                T my = fmax(fmax(fmax(Ml, Dl), fmax(Mul, Dul)), fmax(Iin, acc));
#pragma unroll
                for (int j = 0; j < NR; ++j)
                    my = fmax(my, fmax(M[j], D[j]));
                const int e_my = my > (T)0 ? S::ilogb(my) : kNone;
                const int e = e_in > e_my ? e_in : e_my;
                if (e > kNone && (e > 96 || e < -32))
                    rescale(64 - e);
            };
            auto expo = [&](T v, int e) { return v > (T)0 ? S::ilogb(v) + e : kNone; };
            for (int s = 0; s < nsteps; ++s) {
                const int c = s - lane;  // this lane's 0-based column
                const int letter = (c >= 0 && c < HL)
                                       ? (raw ? (int)bd.hap_data[hoff + c] : (int)p.hapc[hoff + c])
                                       : wild;
                T mp = Mul, dp = Dul, chain = Iin;
                if (lane == 0 && !top) {
                    // row above the tile at column c-1, from the previous tile
                    // (only columns the previous tile wrote: c-1 < HL)
                    if (c >= 1 && c - 1 < HL) {
                        const int emd = ex[2 * (c - 1)] - sc, ei = ex[2 * (c - 1) + 1] - sc;
                        const T rm = sp[3 * (c - 1) + 0], ri = sp[3 * (c - 1) + 1];
                        const T rd = sp[3 * (c - 1) + 2];
                        int e_in = expo(rm, emd);
                        const int e2 = expo(rd, emd), e3 = expo(ri, ei);
                        e_in = e2 > e_in ? e2 : e_in;
                        e_in = e3 > e_in ? e3 : e_in;
                        fit(e_in);
                        const int emd2 = ex[2 * (c - 1)] - sc, ei2 = ex[2 * (c - 1) + 1] - sc;
                        mp = S::ldexp(rm, emd2);
                        chain = S::ldexp(ri, ei2);
                        dp = S::ldexp(rd, emd2);
                    } else {
                        mp = chain = dp = 0;
                    }
                }
#pragma unroll
                for (int j = 0; j < NR; ++j) {
                    const T mo = M[j], dov = D[j];
                    const T lam = (letter == code[j] || letter == wild) ? lm[j] : lx[j];
                    M[j] = lam * (ca[j] * mp + cb[j] * (chain + dp));
                    chain = cdl[j] * mp + ce[j] * chain;
                    // past the read (ce = 1, cs = 0) D stays at its start, 0
                    D[j] = cs[j] * mo + ce[j] * dov;
                    mp = mo;
                    dp = dov;
                }
                if (lane == tr && c >= 1 && c <= HL)
                    acc += chain;
                if (c == HL) {
                    acc_end = acc;
                    sc_end = sc;
                }
                if (!last_tile && lane == 63) {
                    if (c >= 0 && c < HL) {
                        sp[3 * c + 0] = M[NR - 1];
                        sp[3 * c + 2] = D[NR - 1];
                        ex[2 * c] = sc;
                    }
                    if (c >= 1 && c <= HL) {
                        sp[3 * (c - 1) + 1] = chain;
                        ex[2 * (c - 1) + 1] = sc;
                    }
                }
                const T sM = S::shr(M[NR - 1]);
                const T sD = S::shr(D[NR - 1]);
                const T sI = S::shr(chain);
                const int ssc = shr1i(sc);
                if (lane != 0) {
                    int e_in = expo(sM, ssc - sc);
                    const int e2 = expo(sD, ssc - sc), e3 = expo(sI, ssc - sc);
                    e_in = e2 > e_in ? e2 : e_in;
                    e_in = e3 > e_in ? e3 : e_in;
                    fit(e_in);
                } else {
                    fit(kNone);
                }
                const int d = ssc - sc;
                Mul = Ml;
                Dul = Dl;
                Ml = lane == 0 ? (T)0 : S::ldexp(sM, d);
                Dl = lane == 0 ? (top ? C0s : (T)0) : S::ldexp(sD, d);
                Iin = lane == 0 ? (T)0 : S::ldexp(sI, d);
            }
            __syncthreads();  // spilled row visible to the next tile
        }
        // the result lane of the last tile owns the sum
        const int tr = (L - (ntiles - 1) * TR) / NR;
        if (lane == tr) {
            const double lg = log10((double)acc_end) + (double)sc_end * 0.30102999566398119521 -
                              log10((double)C0 * (double)HL);
            bd.scores[it.out] = (float)lg;
            // same criterion as the tile kernels: the sum in the reference's
            // units (start FLT_MAX/16/H) below rescue_min, or not finite
            const double lmin = log10((double)p.rescue_min) - (double)kLog10Scale;
            if (sizeof(T) == 4 && p.rescue_on && !(acc_end > (T)0 && lg >= lmin && lg < 1e30)) {
                const int q = atomicAdd(p.final_count, 1);
                p.final_items[q] = it;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// k_fwd_special
// ---------------------------------------------------------------------------
// What the tile bins cannot take: reads of several tiles (strips) and haps
// holding the wildcard.
//
// Strips: one wave per alignment, the read cut into tiles of 64 lanes x
// kStripRows rows swept one after another with the tile sweep's arithmetic.  A
// tile's last lane writes its last row's (M, I) per column to a border row in
// global memory; the next tile's first lane takes them in instead of row 0 and
// forms D, a chain along the row, itself.  Sixteen columns are read at a time,
// ahead of their use, one per lane, and broadcast from there.  The border row is
// written 64 columns behind where it is read, so the tiles of a read share one.
// The emission table holds the wildcard as a fifth letter.
//
// In FP64 from the start: a deletion's run decays within one lane, so in FP32
// one of 80 bases is flushed whatever the lane's scale, and the long flanks on
// either side of it then cost hundreds in log10 (a 1,200-base read against a
// hap with 80 more bases: -86.5, and -597 in scaled FP32; up to 70 is exact).
// Scores of long reads are mostly below the FP32 range anyway.  A lane's
// power-of-two scale only ever raises what it holds: a score above -596 (2^94
// above double's least value in an unscaled lane, while all that is flushed is
// less than that value per cell) is as good as double is; below, a lane's
// range under its largest value is 2^1274, the wave kernel's is 2^1042.
//
// Bound by the VALU, whose FP64 instructions take four cycles each.  2,560
// alignments of 1100-1500-base reads with 1500-2000-base haps, whole calls: the
// one-wave kernel, with 1024-row tiles, an exponent check of every row per
// column in FP32 and FP64 for what falls below its range, 23.2 ms; scaled FP32
// strips 1.5 ms; these 2.2 ms (without a scale, and the wave kernel for all
// below -596, 1.96 ms, or 5 to 10 ms where a call has such scores).  8 rows per
// lane keep the emission table at 20 KiB, eight blocks per CU, and waste less
// of a read's last tile than 10.
//
// Wildcard haps: the one-wave kernel's arithmetic with as many alignments side
// by side on the wave as its lanes hold, the emission values from an LDS table
// of five letters instead of compares, and the letters loaded four columns
// ahead.  The items are sorted by (read class, hap length) and a wave takes a
// run of them.  908k mixed alignments of which 5% have such a hap: 20.0 -> 7.1
// ms per call.
// Border entries: the longest hap's columns, four exponents each for 64 of them,
// and kStripPad.
constexpr int kStripPad = 256;
// A strip's lane holds its values times 2^E, E >= 0: every 16 columns, where
// the largest of them has left 2^kStripLow .. 2^kStripHigh, E puts it at
// 2^kStripAim again (not below 0).  Between two checks values grow by 2^13 and
// the gap extension per column at most (see kDsEvery), far less than what is
// left above 2^kStripHigh.
constexpr int kStripEvery = 16, kStripLow = 200, kStripAim = 600, kStripHigh = 700;
constexpr int kStripSpan = 1000;  // largest |E_t - E_{t-1}|
// The smallest sum that a strip finishes, in its lane's scale.
constexpr double kStripMin = 0x1p-900;

// Lane `src`'s value, in scalar registers.
__device__ __forceinline__ double lane_value(double v, int src)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), src),
                            __builtin_amdgcn_readlane(__double2loint(v), src));
}

// Every lane's `v` moves one lane down; the last lane takes `top`.
__device__ __forceinline__ double push_top(double v, double top)
{
    // DPP wave_shl:1, the last lane, without a source, keeps `top`
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(top), __double2loint(v), 0x130, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(top), __double2hiint(v), 0x130, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// One alignment on the whole wave; border: the block's border row, which ends
// with lane 63's exponent for every 16 columns.  Returns 1 when the sum is below
// the rescue threshold and finished.
template <bool FAST>
__device__ __forceinline__ int strip_task(const FwdParams& p, double2* tab, double2* border,
                                           const WorkItem& it)
{
    using TT = TileTraits<double>;
    constexpr int NR = kStripRows, NL = 5, TR = kStripTileRows, K = TT::K;
    using Shape = TabShape<double, NR, NL>;
    using S = WaveScalar<double>;
    constexpr int NV = Shape::NV;
    static_assert(!Shape::kTail && NR % K == 0, "whole vectors");
    const BatchDesc& bd = *p.bd;
    const int t = threadIdx.x;
    const bool first = t == 0;
    const double f = first ? 1.0 : 0.0;  // what enters from above, in the first lane only
    const int L = bd.read_len[it.read], HL = bd.hap_len[it.hap];
    const int ntiles = (L + TR) / TR;  // tiles of the read's rows and one more
    const uint32_t* hdw = reinterpret_cast<const uint32_t*>(p.hapc + bd.hap_off[it.hap]);
    const int hdw_last = HL >> 2;
    const uint32_t shift = (uint32_t)(-t) & 3u;
    // (columns outside the hap take some letter of it, or the padding's base 0:
    // nothing of theirs is used)
    auto hap_dword = [&](int q) { return hdw[min(max(q, 0), hdw_last)]; };
    // FAST: nl only scales the start, where its rounding does not matter
    const double scale = FAST ? 0.5 * (double)p.meta[it.read].nl : 1.0;
    const double C0 = kStartF64 / (double)HL * scale;
    const float log2_c0 = (float)log2(C0);
    int32_t* border_exp = reinterpret_cast<int32_t*>(border + HL + 128);

    TileRead<double, NR, false> R;
    double prod = 1.0, sum = 0.0;  // sum: the result lane's, times 2^sum_E
    int E = 0, sum_E = 0;
    bool bad = false;
    for (int k = 0; k < ntiles; ++k) {
        const int row0 = k * TR;
        const bool top = k == 0, last = k == ntiles - 1;
        tile_setup<double, NR, FAST, false, NL>(p, tab, true, it.read, t, R, row0);
        prod *= R.prod;
        // border columns c0 .. c0+15 in lanes 0-15; row 0 has D = C0 in every
        // column, and column HL still carries the chain of the last one (a
        // row's chain runs one column behind)
        auto fetch = [&](int c0) {
            const int c = c0 + t;
            return top || t >= 16 || c > HL ? make_double2(0.0, 0.0) : border[64 + c];
        };
        const int res_t = last ? (L - row0) / NR : 63;
        // a lane's first values are those of the insertion floor (see kDsFloor)
        E = top && first ? 0 : max(0, kStripAim - (int)floorf(log2_c0 + R.floor2));
        double nf;  // what the lane above is multiplied by
        auto set_factor = [&]() {
            const int d = E - ds_above(E);
            bad = bad || (!first && t <= res_t && (d > kStripSpan || d < -kStripSpan));
            nf = first ? 0.0 : ldexp(1.0, d);
        };
        set_factor();
        // the exponent of the 16 columns up to 16 b - 48, and a fetched value on
        // the first lane's
        auto fetch_exp = [&](int b) { return top ? 0 : border_exp[b]; };
        auto scaled = [&](const double2& v, int e) {
            const int sh = __builtin_amdgcn_readfirstlane(E) - e;
            return make_double2(ldexp(v.x, sh), ldexp(v.y, sh));
        };
        typename TT::P MD[NR], MDr[2];
#pragma unroll
        for (int j = 0; j < NR; ++j)
            MD[j] = 0.0;
        // before step 0 the first lane holds the row above at columns -1 (row
        // 0 only) and 0
        const double2 b0 = scaled(fetch(0), fetch_exp(3));
        const double eb = top ? 1.0 : R.eps;
        double Ma = lane_value(b0.x, 0), Da = top ? C0 : 0.0;  // the row above's last M and D
        MDr[0].x = 0.0;
        MDr[0].y = f * Da;
        MDr[1].x = f * Ma;
        MDr[1].y = f * Da;
        double Iin = f * lane_value(b0.y, 0);
        double2 raw = fetch(1);
        int raw_exp = fetch_exp(4);
        double2 out = make_double2(0.0, 0.0);  // the last 16 columns of the last row, lanes 48-63
        double acc = 0.0;
        sum = 0.0;
        sum_E = E;
        const int nsteps = HL + res_t + 1;
        const int acc_last = t + HL;

        const int q0 = (0 - t) >> 2;
        uint32_t wlo = hap_dword(q0), whi = hap_dword(q0 + 1), wnx = hap_dword(q0 + 2);
        uint32_t letters = __builtin_amdgcn_alignbyte(whi, wlo, shift);
        double2 lam[2][NV];
#pragma unroll
        for (int q = 0; q < NV; ++q)
            lam[0][q] = (tab + (((letters & 7u) << 6) | t))[q * (NL * 64)];
        auto sweep4 = [&](int s4, int w4, const double2& win, bool bounded) {
            const uint32_t next = __builtin_amdgcn_alignbyte(wnx, whi, shift);
            const uint32_t wn2 = hap_dword(((s4 - t) >> 2) + 3);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int cur = u & 1, nxt = cur ^ 1;
                const uint32_t nletter = u < 3 ? (letters >> (8 * (u + 1))) & 7u : next & 7u;
                const double2* trow = tab + ((nletter << 6) | t);
#pragma unroll
                for (int q = 0; q < NV; ++q)
                    lam[nxt][q] = trow[q * (NL * 64)];
                // the row above at column s + 1
                const double in_m = lane_value(win.x, w4 + u), in_i = lane_value(win.y, w4 + u);
                Da = fma(eb, Da, Ma);
                Ma = in_m;
                TT::P up = MDr[cur];
                double chain = Iin;
#pragma unroll
                for (int q = 0; q < NV; ++q) {
                    double lv[K];
                    TT::unpack(lam[cur][q], lv);
#pragma unroll
                    for (int x = 0; x < K; ++x)
                        tile_cell<double, NR, FAST, false>(R, K * q + x, lv[x], R.eps, MD[K * q + x],
                                                           up, chain);
                }
                if (bounded)
                    acc += (s4 + u <= acc_last) ? chain : 0.0;
                else
                    acc += chain;
                out.x = push_top(out.x, MD[NR - 1].x);
                out.y = push_top(out.y, chain);
                __builtin_amdgcn_s_setprio(3);  // as in tile_sweep
                MDr[cur].x = fma(f, in_m, shr1d(MD[NR - 1].x) * nf);
                MDr[cur].y = fma(f, Da, shr1d(MD[NR - 1].y) * nf);
                Iin = fma(f, in_i, shr1d(chain) * nf);
                __builtin_amdgcn_s_setprio(0);
            }
            letters = next;
            wlo = whi;
            whi = wnx;
            wnx = wn2;
        };
        static_assert(kStripEvery == 16, "one window between two checks");
        for (int s0 = 0; s0 < nsteps; s0 += 16) {
            // columns s0+1 .. s0+16 for the steps below; the next 16 are
            // fetched over them
            const double2 win = scaled(raw, raw_exp);
            raw = fetch(s0 + 17);
            raw_exp = fetch_exp((s0 >> 4) + 5);
            if (s0 + 16 <= HL + 1) {
#pragma unroll
                for (int w4 = 0; w4 < 16; w4 += 4)
                    sweep4(s0 + w4, w4, win, false);
            } else {
                for (int w4 = 0; w4 < 16; w4 += 4)
                    sweep4(s0 + w4, w4, win, true);
            }
            if (!last && t >= 48)  // columns s0 - 63 .. s0 - 48
                border[s0 + 1 + t - 48] = out;
            if (!last && t == 63)
                border_exp[s0 >> 4] = E;
            // the sum on the larger value's scale, so that it does not hold back
            // the lane's own
            const int lower = min(sum_E, E);
            sum = ldexp(sum, lower - sum_E) + ldexp(acc, lower - E);
            sum_E = lower;
            acc = 0.0;
            double my = fmax(fmax(fmax(MDr[0].x, MDr[0].y), fmax(MDr[1].x, MDr[1].y)), Iin);
#pragma unroll
            for (int j = 0; j < NR; ++j)
                my = fmax(my, fmax(MD[j].x, MD[j].y));
            const int e = S::expo(my);
            int x = E;
            if (my > 0.0 && (e < kStripLow || (e > kStripHigh && E > 0)))
                x = max(0, E + kStripAim - e);
            if (__ballot(x != E)) {
                const int sh = x - E;
#pragma unroll
                for (int j = 0; j < NR; ++j) {
                    MD[j].x = ldexp(MD[j].x, sh);
                    MD[j].y = ldexp(MD[j].y, sh);
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    MDr[u].x = ldexp(MDr[u].x, sh);
                    MDr[u].y = ldexp(MDr[u].y, sh);
                }
                Iin = ldexp(Iin, sh);
                const int sh0 = __builtin_amdgcn_readfirstlane(sh);
                Ma = ldexp(Ma, sh0);
                Da = ldexp(Da, sh0);
                E = x;
                set_factor();
            }
        }
        __syncthreads();  // the border row is visible to the next tile
    }
    double lp = FAST ? log10(prod) : 0.0;
    if (FAST) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            lp += __shfl_xor(lp, o, 64);
    }
    const bool ok = __ballot(bad) == 0;
    bool done = false;
    if (t == (L - (ntiles - 1) * TR) / NR) {
        const double lg = log10(sum) - (double)sum_E * 0.30102999566398119521 +
                          (FAST ? lp - log10(scale) : -log10(R.beta)) - kLog10StartF64;
        bd.scores[it.out] = (float)lg;
        // gap scores too steep for the checks: the wave kernel checks every step
        if (!(ok && sum >= kStripMin && sum < 0x1p1020))
            p.final_items[atomicAdd(p.final_count, 1)] = it;
        else
            done = lg < log10((double)p.rescue_min) - kLog10ScaleD;
    }
    return __ballot(done) ? 1 : 0;
}

// LDS of both (20 KiB, so that eight blocks share a CU): the wildcard tiles'
// emission table or a strip's.
union SpecialTab {
    float4 f32[TabShape<float, kWildRows, 5>::kWords];
    double2 f64[TabShape<double, kStripRows, 5>::kWords];
};
static_assert(sizeof(SpecialTab) <= 20 << 10, "eight blocks per CU");

// Items per wildcard task: 12 or 24 fill whole waves for most reads (4, 6 or
// 12 side by side); the longer run where every wave gets several, the shorter
// (or, for few items, 4) to spread them over the device.  Runs of 4 / 12 / 24,
// us per call of wildcard haps only, by items per wave: 3.8: 817 / 1294 / 2190,
// 40: 3257 / 3014 / 3594, 132: 8951 / 8182 / 8159, 295: 18995 / 16711 / 16451.
__device__ __forceinline__ int wild_run(int nw)
{
    const int per_wave = nw / (int)gridDim.x;
    return per_wave >= 72 ? 24 : per_wave >= 4 ? 12 : 4;
}
// The block's border row; returns how many of the launch's first blocks the
// arena holds one for (none: the first block reports it).  Its length is that
// of the longest hap that a strip meets, so that a batch's other haps cost the
// strips no blocks.
__device__ __forceinline__ int border_row(const SpecialSet& ss, double2*& border)
{
    const int64_t stride = (int64_t)*ss.hmax + (*ss.hmax >> 6) + kStripPad;
    const int64_t rows = ss.border_entries / stride;
    if (rows <= 0 && blockIdx.x == 0 && threadIdx.x == 0)
        *(volatile int32_t*)ss.error_flag = 1;
    border = ss.border + blockIdx.x * stride;
    return (int)(rows < (int64_t)gridDim.x ? rows : (int64_t)gridDim.x);
}
// A launch's strips (nm > 0), one each per task, on the blocks that have a
// border row.  They come before the launch's other tasks: a strip takes longest,
// and the blocks without a border row start on the others at once.  (57,600
// alignments of 150-base reads with 4 and with 300 of 1,100 bases, where the
// others came first and on the blocks with a border row only: 1167 -> 860 and
// 1298 -> 983 us.)
__device__ __forceinline__ int strip_tasks(const FwdParams& p, const SpecialSet& ss, SpecialTab& tab,
                                           const WorkItem* strips, int nm)
{
    double2* border = nullptr;
    const int blocks = border_row(ss, border);
    if ((int)blockIdx.x >= blocks)
        return 0;
    int done = 0;
    for (int task = next_task(ss.next_strip, nm, blocks, true); task < nm;
         task = next_task(ss.next_strip, nm, blocks, false)) {
        const WorkItem it = strips[__builtin_amdgcn_readfirstlane(task)];
        const ReadMeta m = p.meta[it.read];
        const bool fast = m.bin == ss.strip_bin ? m.nl > 0.f : (m.bin & 1) == 0;
        done += fast ? strip_task<true>(p, tab.f64, border, it)
                     : strip_task<false>(p, tab.f64, border, it);
    }
    return done;
}
// The next of the launch's other tasks.  Where there are strips, no block has
// one of its own, which a strip would hold back.
__device__ __forceinline__ int next_other(const SpecialSet& ss, int total, bool strips, bool first)
{
    return strips ? counter_task(ss.next_task) : next_task(ss.next_task, total, gridDim.x, first);
}
// Run `q` of the wildcard items.
__device__ __forceinline__ void wild_task(const FwdParams& p, SpecialTab& tab, const WorkItem* wilds,
                                          int nw, int run, int q)
{
    int i = q * run;
    const int end = min(i + run, nw);
    while (i < end) {  // as many of the next items as fit side by side
        const int n = end - i;  // at most 24: one lane each
        const int L = (int)threadIdx.x < n ? p.bd->read_len[wilds[i + threadIdx.x].read] : 0;
        const int G = (wave_max(L) + kWildRows) / kWildRows;  // ceil((L + 1) / rows)
        const int take = min(n, 64 / G);
        pack_task<float, kWildRows>(p, tab.f32, wilds + i, take, G);
        i += take;
    }
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 8))) void k_fwd_special(
    FwdParams p, SpecialSet ss)
{
    __shared__ SpecialTab tab;
    const int nm = ss.range[2 * ss.strip_bin + 1], nw = ss.range[2 * ss.wild_bin + 1];
    if (nm + nw == 0)
        return;
    const WorkItem* strips = ss.items + ss.range[2 * ss.strip_bin];
    const WorkItem* wilds = ss.items + ss.range[2 * ss.wild_bin];
    const BatchDesc bd = *p.bd;
    p.bd = &bd;
    const int done = nm > 0 ? strip_tasks(p, ss, tab, strips, nm) : 0;
    const int run = wild_run(nw);
    const int total = (nw + run - 1) / run;
    for (int task = next_other(ss, total, nm > 0, true); task < total;
         task = next_other(ss, total, nm > 0, false))
        wild_task(p, tab, wilds, nw, run, __builtin_amdgcn_readfirstlane(task));
    if (done > 0 && threadIdx.x == 0)
        atomicAdd(p.scaled_total, (unsigned long long)done);
}

// The FP32 pass of a small call in one launch: the strips, then FAST
// super-tasks, SAFE ones and wildcard items, in that order from one counter.
template <bool GE>
__device__ __forceinline__ int tiny_tasks(const FwdParams& p, const SpecialSet& ss,
                                          const TinyLists& tl, SpecialTab& tab, bool strips)
{
    const int nf = tl.counts[kTinyFast], ns = tl.counts[kTinySafe], nw = tl.counts[kTinyWilds];
    const int run = wild_run(nw);
    const int total = nf + ns + (nw + run - 1) / run;
    int done = 0;
    for (int task = next_other(ss, total, strips, true); task < total;
         task = next_other(ss, total, strips, false)) {
        task = __builtin_amdgcn_readfirstlane(task);
        if (task < nf + ns) {
            const bool fast = task < nf;
            const SuperTask st = fast ? tl.st[0][task] : tl.st[1][task - nf];
            const int G = __builtin_amdgcn_readfirstlane(st.nc >> 8);
            // what the scaling refuses: the FP64 tiles hold 512 rows, the
            // classes above them have more than 32 lanes
            FwdParams q = p;
            const bool tiles = G <= 512 / kTinyRows;
            q.rescue_items = !tiles ? p.final_items : fast ? tl.rescue[0] : tl.rescue[1];
            q.rescue_counts = !tiles ? p.final_count
                                     : tl.counts + (fast ? kTinyRescueFast : kTinyRescueSafe);
            done += fast ? tile_super_task<float, kTinyRows, true, false, true, GE>(q, tab.f32, st, G, 0, 0)
                         : tile_super_task<float, kTinyRows, false, false, true, GE>(q, tab.f32, st, G, 0, 0);
        } else {
            wild_task(p, tab, tl.wilds, nw, run, task - nf - ns);
        }
    }
    return done;
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 8))) void k_fwd_tiny(
    FwdParams p, SpecialSet ss, TinyLists tl)
{
    static_assert(TabShape<float, kTinyRows>::kWords <= TabShape<float, kWildRows, 5>::kWords,
                  "one table for all");
    __shared__ SpecialTab tab;
    const BatchDesc bd = *p.bd;
    p.bd = &bd;
    const int nm = tl.counts[kTinyStrips];
    int done = nm > 0 ? strip_tasks(p, ss, tab, tl.strips, nm) : 0;
    done += p.semantics == 0 ? tiny_tasks<true>(p, ss, tl, tab, nm > 0)
                             : tiny_tasks<false>(p, ss, tl, tab, nm > 0);
    if (done > 0 && threadIdx.x == 0)
        atomicAdd(p.scaled_total, (unsigned long long)done);
}

// FP64 recompute of a small call's rescue lists, usually empty: the 10-row
// FAST and 8-row SAFE tiles (the rows of the small-batch table's FP64 sets),
// runs of a few items per wave.  What they cannot finish joins the late list.
template <int NR, bool FAST>
__device__ __forceinline__ void rescue_list(const FwdParams& p, double2* tab, const WorkItem* items,
                                            int n)
{
    constexpr int kRun = 6;
    for (int v = blockIdx.x * kRun; v < n; v += gridDim.x * kRun) {
        const int end = min(n, v + kRun);
        for (int i = v; i < end;) {
            const int rem = end - i;
            const int L = (int)threadIdx.x < rem ? p.bd->read_len[items[i + threadIdx.x].read] : 0;
            const int G = (wave_max(L) + NR) / NR;  // ceil((L + 1) / NR)
            const int take = min(rem, 64 / G);
            tile_items_task<double, NR, FAST, false>(p, tab, items, i, take, G, 0, 0, 0);
            i += take;
        }
    }
}
__global__ __launch_bounds__(64) void k_rescue_tiny(FwdParams p, TinyLists tl, int64_t* totals)
{
    __shared__ double2 tab[TabShape<double, 10>::kWords];
    const int nf = tl.counts[kTinyRescueFast], ns = tl.counts[kTinyRescueSafe];
    if (nf + ns == 0)
        return;
    if (blockIdx.x == 0 && threadIdx.x < 2)
        atomicAdd(reinterpret_cast<unsigned long long*>(totals + threadIdx.x),
                  (unsigned long long)(nf + ns));
    p.final_items = tl.late;
    p.final_count = tl.counts + kTinyLate;
    rescue_list<10, true>(p, tab, tl.rescue[0], nf);
    rescue_list<8, false>(p, tab, tl.rescue[1], ns);
}

hipError_t launch_rescue_tiny(const FwdParams& p, const TinyLists& tl, int grid, int64_t* totals,
                              hipStream_t st)
{
    hipLaunchKernelGGL(k_rescue_tiny, dim3(grid), dim3(64), 0, st, p, tl, totals);
    return hipGetLastError();
}

hipError_t launch_fwd_tiny(const FwdParams& p, const SpecialSet& ss, const TinyLists& tl, int grid,
                           hipStream_t st)
{
    if (!p.scaled_total || !p.rescue_on || !ss.next_task || !ss.next_strip || !ss.hmax || !ss.border ||
        !ss.error_flag || grid <= 0)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_fwd_tiny, dim3(grid), dim3(64), 0, st, p, ss, tl);
    return hipGetLastError();
}

hipError_t launch_fwd_special(const FwdParams& p, const SpecialSet& ss, int grid, hipStream_t st)
{
    if (!p.scaled_total || !p.rescue_on || !ss.items || !ss.range || !ss.next_task || !ss.next_strip || !ss.hmax ||
        !ss.border || !ss.error_flag || grid <= 0)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_fwd_special, dim3(grid), dim3(64), 0, st, p, ss);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
template <typename K>
static int resident_blocks_per_cu(K kernel)
{
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, 64, 0) != hipSuccess) {
        (void)hipGetLastError();
        n = 0;
    }
    return n > 0 ? n : 4;
}

template <typename T, int NR, bool FAST, bool ROWEPS = false, bool RE = false, bool DS = false>
static int set_blocks_per_cu()
{
    static const int n = resident_blocks_per_cu(k_fwd_tile_set<T, NR, FAST, ROWEPS, RE, DS>);
    return n;
}

static int grid_of(int grid, int per_cu)
{
    if (grid > 0)
        return grid;
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
            cus = prop.multiProcessorCount;
        else {
            (void)hipGetLastError();
            cus = 256;
        }
    }
    return cus * per_cu;
}

template <typename T, int NR, bool ROWEPS = false, bool RE = false, bool DS = false>
static hipError_t launch_set_nr(bool fast, const FwdParams& p, const BinSet& bs, int grid,
                                hipStream_t st)
{
    if (bs.n < 1 || bs.n > 64 || !bs.counts || !bs.next_task || (!bs.items && !bs.st))
        return hipErrorInvalidValue;
    if (RE && (bs.st || !bs.seg || !p.retry_items || !p.retry_counts || !p.rescue_exps))
        return hipErrorInvalidValue;
    if (DS && (!p.scaled_total || !p.rescue_on))
        return hipErrorInvalidValue;
    for (int i = 0; i < bs.n; ++i)
        if (bs.lanes[i] < 1 || bs.lanes[i] > 64)
            return hipErrorInvalidValue;
    if (fast) {
        hipLaunchKernelGGL((k_fwd_tile_set<T, NR, true, ROWEPS, RE, DS>),
                           dim3(grid_of(grid, set_blocks_per_cu<T, NR, true, ROWEPS, RE, DS>())),
                           dim3(64), 0, st, p, bs);
    } else {
        hipLaunchKernelGGL((k_fwd_tile_set<T, NR, false, ROWEPS, RE, DS>),
                           dim3(grid_of(grid, set_blocks_per_cu<T, NR, false, ROWEPS, RE, DS>())),
                           dim3(64), 0, st, p, bs);
    }
    return hipGetLastError();
}

bool tile_re_supported(int NR) { return re_rows(NR); }

hipError_t launch_fwd_tile_set_re(int NR, bool fast, const FwdParams& p, const BinSet& bs,
                                  int grid, hipStream_t st)
{
    switch (NR) {
    case 12: return launch_set_nr<float, 12, false, true>(fast, p, bs, grid, st);
    case 13: return launch_set_nr<float, 13, false, true>(fast, p, bs, grid, st);
    case 16: return launch_set_nr<float, 16, false, true>(fast, p, bs, grid, st);
    case 19: return launch_set_nr<float, 19, false, true>(fast, p, bs, grid, st);
    case 20: return launch_set_nr<float, 20, false, true>(fast, p, bs, grid, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_fwd_tile_set_scaled(int NR, bool fast, const FwdParams& p, const BinSet& bs,
                                      int grid, hipStream_t st)
{
    switch (NR) {
    case 12: return launch_set_nr<float, 12, false, false, true>(fast, p, bs, grid, st);
    case 13: return launch_set_nr<float, 13, false, false, true>(fast, p, bs, grid, st);
    case 16: return launch_set_nr<float, 16, false, false, true>(fast, p, bs, grid, st);
    case 19: return launch_set_nr<float, 19, false, false, true>(fast, p, bs, grid, st);
    case 20: return launch_set_nr<float, 20, false, false, true>(fast, p, bs, grid, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_fwd_tile_set(int NR, bool fast, const FwdParams& p, const BinSet& bs, int grid,
                               hipStream_t st, bool roweps)
{
    if (roweps)  // per-position gcp: the 16-row tiles only
        return NR == kRowEpsRows32 ? launch_set_nr<float, kRowEpsRows32, true>(fast, p, bs, grid, st)
                                   : hipErrorInvalidValue;
    switch (NR) {
    case 4: return launch_set_nr<float, 4>(fast, p, bs, grid, st);
    case 8: return launch_set_nr<float, 8>(fast, p, bs, grid, st);
    case 12: return launch_set_nr<float, 12>(fast, p, bs, grid, st);
    case 13: return launch_set_nr<float, 13>(fast, p, bs, grid, st);
    case 16: return launch_set_nr<float, 16>(fast, p, bs, grid, st);
    case 19: return launch_set_nr<float, 19>(fast, p, bs, grid, st);
    case 20: return launch_set_nr<float, 20>(fast, p, bs, grid, st);
    case 24: return launch_set_nr<float, 24>(fast, p, bs, grid, st);
    case 28: return launch_set_nr<float, 28>(fast, p, bs, grid, st);
    case 32: return launch_set_nr<float, 32>(fast, p, bs, grid, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_fwd_tile_set_f64(int NR, bool fast, const FwdParams& p, const BinSet& bs,
                                   int grid, hipStream_t st, bool roweps)
{
    if (roweps)  // per-position gcp: the 8-row FP64 tiles only
        return NR == kRowEpsRows64 ? launch_set_nr<double, kRowEpsRows64, true>(fast, p, bs, grid, st)
                                   : hipErrorInvalidValue;
    switch (NR) {
    case 4: return launch_set_nr<double, 4>(fast, p, bs, grid, st);
    case 6: return launch_set_nr<double, 6>(fast, p, bs, grid, st);
    case 8: return launch_set_nr<double, 8>(fast, p, bs, grid, st);
    case 10: return launch_set_nr<double, 10>(fast, p, bs, grid, st);
    default: return hipErrorInvalidValue;
    }
}

int tile_set_blocks_per_cu(int NR, bool fast, bool f64, bool roweps, bool scaled)
{
    if (scaled && !f64 && !roweps) {
        switch (NR) {
        case 12: return fast ? set_blocks_per_cu<float, 12, true, false, false, true>()
                             : set_blocks_per_cu<float, 12, false, false, false, true>();
        case 13: return fast ? set_blocks_per_cu<float, 13, true, false, false, true>()
                             : set_blocks_per_cu<float, 13, false, false, false, true>();
        case 16: return fast ? set_blocks_per_cu<float, 16, true, false, false, true>()
                             : set_blocks_per_cu<float, 16, false, false, false, true>();
        case 19: return fast ? set_blocks_per_cu<float, 19, true, false, false, true>()
                             : set_blocks_per_cu<float, 19, false, false, false, true>();
        case 20: return fast ? set_blocks_per_cu<float, 20, true, false, false, true>()
                             : set_blocks_per_cu<float, 20, false, false, false, true>();
        default: return 0;
        }
    }
    if (roweps) {
        if (!f64 && NR == kRowEpsRows32)
            return fast ? set_blocks_per_cu<float, kRowEpsRows32, true, true>()
                        : set_blocks_per_cu<float, kRowEpsRows32, false, true>();
        if (f64 && NR == kRowEpsRows64)
            return fast ? set_blocks_per_cu<double, kRowEpsRows64, true, true>()
                        : set_blocks_per_cu<double, kRowEpsRows64, false, true>();
        return 0;
    }
    if (f64) {
        switch (NR) {
        case 4: return fast ? set_blocks_per_cu<double, 4, true>() : set_blocks_per_cu<double, 4, false>();
        case 6: return fast ? set_blocks_per_cu<double, 6, true>() : set_blocks_per_cu<double, 6, false>();
        case 8: return fast ? set_blocks_per_cu<double, 8, true>() : set_blocks_per_cu<double, 8, false>();
        case 10: return fast ? set_blocks_per_cu<double, 10, true>() : set_blocks_per_cu<double, 10, false>();
        default: return 0;
        }
    }
    switch (NR) {
    case 4: return fast ? set_blocks_per_cu<float, 4, true>() : set_blocks_per_cu<float, 4, false>();
    case 8: return fast ? set_blocks_per_cu<float, 8, true>() : set_blocks_per_cu<float, 8, false>();
    case 12: return fast ? set_blocks_per_cu<float, 12, true>() : set_blocks_per_cu<float, 12, false>();
    case 13: return fast ? set_blocks_per_cu<float, 13, true>() : set_blocks_per_cu<float, 13, false>();
    case 16: return fast ? set_blocks_per_cu<float, 16, true>() : set_blocks_per_cu<float, 16, false>();
    case 19: return fast ? set_blocks_per_cu<float, 19, true>() : set_blocks_per_cu<float, 19, false>();
    case 20: return fast ? set_blocks_per_cu<float, 20, true>() : set_blocks_per_cu<float, 20, false>();
    case 24: return fast ? set_blocks_per_cu<float, 24, true>() : set_blocks_per_cu<float, 24, false>();
    case 28: return fast ? set_blocks_per_cu<float, 28, true>() : set_blocks_per_cu<float, 28, false>();
    case 32: return fast ? set_blocks_per_cu<float, 32, true>() : set_blocks_per_cu<float, 32, false>();
    default: return 0;
    }
}

hipError_t launch_fwd_wave_f32(const FwdParams& p, const BinSet& bs, const int32_t* hmax_ptr,
                               float* spill, int64_t spill_elems, int32_t* error_flag, int blocks,
                               hipStream_t st)
{
    if (bs.n < 1 || bs.n > 64 || !bs.counts || !bs.items || blocks <= 0)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_fwd_wave<float, 16>), dim3(blocks), dim3(64), 0, st, p, bs, hmax_ptr,
                       spill, spill_elems, error_flag, (int64_t*)nullptr);
    return hipGetLastError();
}

hipError_t launch_fwd_wave_f64(const FwdParams& p, const BinSet& bs, const int32_t* hmax_ptr,
                               double* spill, int64_t spill_elems, int32_t* error_flag, int blocks,
                               hipStream_t st, bool pack, int64_t* totals)
{
    if (bs.n < 1 || bs.n > 64 || !bs.counts || !bs.items || blocks <= 0)
        return hipErrorInvalidValue;
    if (pack)
        hipLaunchKernelGGL((k_fwd_wave<double, 8, true>), dim3(blocks), dim3(64), 0, st, p, bs,
                           hmax_ptr, spill, spill_elems, error_flag, totals);
    else
        hipLaunchKernelGGL((k_fwd_wave<double, 8>), dim3(blocks), dim3(64), 0, st, p, bs, hmax_ptr,
                           spill, spill_elems, error_flag, totals);
    return hipGetLastError();
}

}  // namespace phmm
