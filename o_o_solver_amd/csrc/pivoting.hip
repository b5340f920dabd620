// The indefinite factorisation with Bunch–Kaufman pivoting: the kernels of the pivoted fronts, and the solve-side
// kernels of a pivoted factor (unit lower block inverses, the 2 × 2 block diagonal, the pivot permutation).
//
// A pivoted front is a full N × N column-major array (leading dimension N, lower triangle used) whose positions are
// [the supernode's own c columns, the d columns its children delayed, its r rows]; the first C = c + d are the
// candidates. Its elimination runs in steps of up to 16 columns: one workgroup per front eliminates them
// (pivotPanelKernel, the rows in registers; pivotColumnsKernel for fronts with more rows than those hold), W = the
// updated columns, L·D; then the candidates to the right get C −= L·Wᵀ by MFMA tiles that read from the front's state
// how far the step got (pivotTrailingKernel), so the host launches a level's steps without waiting for each. After
// the last step the rows below the candidates get the same product with K = e, the eliminated count
// (updateTilesKernel<double, true>). The pivot tests are those of
// src/linalg/kernels/reference/DenseBlockKernels.cpp:448-580: α = (1 + √17)/8, and a candidate whose partner row is
// not a candidate is pivoted alone when |a_kk| >= 0.01·colmax and delayed otherwise (moved behind the candidates still
// to try); passes over the delayed candidates repeat while a pass eliminates something.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

namespace oosg
{

typedef double double4_t __attribute__((ext_vector_type(4)));

namespace
{

constexpr double BK_ALPHA = 0.6403882032022076; // (1 + √17) / 8
constexpr double BK_DELAY = 0.01;                // DenseKernelEntryPoints.hpp:241
constexpr int BK_THREADS = 256;

struct MaxAt
{
    double v;
    int i;
};

// The larger value, the smaller index on a tie: a scan in increasing index order with a strict test keeps the first.
__device__ inline MaxAt larger(MaxAt a, MaxAt b)
{
    return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}

__device__ inline MaxAt blockMax(MaxAt m, double* rv, int* ri)
{
    const int tid = threadIdx.x;
    rv[tid] = m.v;
    ri[tid] = m.i;
    __syncthreads();
    for (int half = BK_THREADS / 2; half > 0; half >>= 1)
    {
        if (tid < half)
        {
            const MaxAt o = larger(MaxAt{rv[tid], ri[tid]}, MaxAt{rv[tid + half], ri[tid + half]});
            rv[tid] = o.v;
            ri[tid] = o.i;
        }
        __syncthreads();
    }
    const MaxAt out{rv[0], ri[0]};
    __syncthreads();
    return out;
}

__device__ inline void swapValues(double& a, double& b)
{
    const double t = a;
    a = b;
    b = t;
}

// W(i, dst) = A(i, col) − Σ_{t ∈ [k0, k)} L(i, t)·W(col, t) for the rows i in [k, N): the column col of the front
// updated by the block's eliminated columns (those before k0 are in the stored values already). A(i, col) is read
// from the lower triangle: column col below its diagonal, row col before it.
__device__ inline void updatedColumn(const double* F, double* W, int N, int k0, int k, int col, int dst, double* wr)
{
    const int tid = threadIdx.x, terms = k - k0;
    for (int t = tid; t < terms; t += BK_THREADS)
        wr[t] = W[col + int64_t(k0 + t) * N];
    __syncthreads();
    for (int i = k + tid; i < N; i += BK_THREADS)
    {
        double a = i >= col ? F[i + int64_t(col) * N] : F[col + int64_t(i) * N];
        for (int t = 0; t < terms; ++t)
            a -= F[i + int64_t(k0 + t) * N] * wr[t];
        W[i + int64_t(dst) * N] = a;
    }
    __syncthreads();
}

// The symmetric interchange of positions p < q of the front (DenseBlockKernels.cpp:69-79), over the stored values:
// rows p and q of the columns before p (the eliminated columns' L, and the columns still to come), the parts between,
// below and on the diagonal; with rows p and q of the block's W columns and the permutation.
template <int THREADS>
__device__ inline void interchange(double* F, double* W, int32_t* perm, int N, int k0, int k, int p, int q)
{
    const int tid = threadIdx.x;
    for (int t = tid; t < p; t += THREADS)
        swapValues(F[p + int64_t(t) * N], F[q + int64_t(t) * N]);
    for (int i = p + 1 + tid; i < q; i += THREADS)
        swapValues(F[i + int64_t(p) * N], F[q + int64_t(i) * N]);
    for (int i = q + 1 + tid; i < N; i += THREADS)
        swapValues(F[i + int64_t(p) * N], F[i + int64_t(q) * N]);
    for (int t = k0 + tid; t < k; t += THREADS)
        swapValues(W[p + int64_t(t) * N], W[q + int64_t(t) * N]);
    if (tid == 0)
    {
        swapValues(F[p + int64_t(p) * N], F[q + int64_t(q) * N]);
        const int32_t e = perm[p];
        perm[p] = perm[q];
        perm[q] = e;
    }
    __syncthreads();
}

// One step of the Bunch–Kaufman elimination of each front of the list (one workgroup per front), for fronts of any
// size: from the front's state, columns are eliminated until `nb` of them are (one more when the last pivot is 2 × 2)
// or the candidates are done, each column computed left-looking from the step's columns in memory. The state records
// where the step started and where the next one does.
//
// Bound by one CU's reads of the step's columns, which grow with their number, against the trailing update's pass over
// the candidates per step. A dense matrix of 5,000 equations (and of 7,000): 261 (508) ms with 64 columns to a step,
// 180 (352) with 32, 142 (280) with 16, 129 (255) with 8, 132 (266) with 4.
__global__ __launch_bounds__(BK_THREADS) void pivotColumnsKernel(const PivotFront* fronts, PivotState* states,
                                                                 const int32_t* list, int nb)
{
    __shared__ double wr[2 * PANEL_BLOCK + 8];
    __shared__ double rv[BK_THREADS];
    __shared__ int ri[BK_THREADS];
    const int q = list[blockIdx.x];
    const PivotFront fr = fronts[q];
    const PivotState st = states[q];
    if (st.done)
    {
        if (threadIdx.x == 0)
            states[q].from = st.k;
        return;
    }
    double* F = fr.F;
    double* W = fr.W;
    int32_t* perm = fr.perm;
    const int N = fr.N, C = fr.C, tid = threadIdx.x;
    const int k0 = st.k;
    int k = st.k, end = st.end, passStart = st.passStart, twoByTwo = st.twoByTwo, done = 0;
    for (;;)
    {
        if (k == end)
        {
            if (end == C || k == passStart)
            {
                done = 1;
                break;
            }
            passStart = k; // another pass over the delayed candidates
            end = C;
            continue;
        }
        if (k - k0 >= nb)
            break;
        updatedColumn(F, W, N, k0, k, k, k, wr);
        const double absakk = fabs(W[k + int64_t(k) * N]);
        MaxAt m{0.0, k};
        for (int i = k + 1 + tid; i < N; i += BK_THREADS)
        {
            const double v = fabs(W[i + int64_t(k) * N]);
            if (v > m.v)
                m = MaxAt{v, i};
        }
        m = blockMax(m, rv, ri);
        const double colmax = m.v;
        const int imax = m.i;
        if (absakk == 0.0 && colmax == 0.0)
        {
            // A zero column: a zero pivot, nothing to eliminate with it.
            for (int i = k + 1 + tid; i < N; i += BK_THREADS)
                F[i + int64_t(k) * N] = 0.0;
            if (tid == 0)
            {
                F[k + int64_t(k) * N] = 0.0;
                fr.diag[k] = 0.0;
                fr.sub[k] = 0.0;
            }
            __syncthreads();
            k += 1;
            continue;
        }
        int blockSize = 1, swapWith = k;
        if (absakk < BK_ALPHA * colmax && imax >= end)
        {
            if (absakk < BK_DELAY * colmax)
            {
                // The partner is not a candidate and the diagonal is too small: delay the column.
                --end;
                if (k != end)
                    interchange<BK_THREADS>(F, W, perm, N, k0, k, k, end);
                continue;
            }
        }
        else if (absakk < BK_ALPHA * colmax)
        {
            // Column imax, updated, in W's column k + 1 (imax < end <= C, so k + 1 < C).
            updatedColumn(F, W, N, k0, k, imax, k + 1, wr);
            double rowmax = 0.0;
            for (int i = k + tid; i < N; i += BK_THREADS)
                if (i != imax)
                    rowmax = fmax(rowmax, fabs(W[i + int64_t(k + 1) * N]));
            rowmax = blockMax(MaxAt{rowmax, 0}, rv, ri).v;
            if (absakk >= BK_ALPHA * colmax * (colmax / rowmax))
                swapWith = k;
            else if (fabs(W[imax + int64_t(k + 1) * N]) >= BK_ALPHA * rowmax)
                swapWith = imax;
            else
            {
                swapWith = imax;
                blockSize = 2;
            }
        }
        const int moved = k + blockSize - 1;
        if (swapWith != moved)
        {
            interchange<BK_THREADS>(F, W, perm, N, k0, k, moved, swapWith);
            if (blockSize == 1)
            {
                // The pivot column is column imax, its rows k and imax exchanged.
                for (int i = k + tid; i < N; i += BK_THREADS)
                {
                    const int from = i == k ? swapWith : (i == swapWith ? k : i);
                    W[i + int64_t(k) * N] = W[from + int64_t(k + 1) * N];
                }
            }
            else if (tid == 0)
            {
                swapValues(W[(k + 1) + int64_t(k) * N], W[swapWith + int64_t(k) * N]);
                swapValues(W[(k + 1) + int64_t(k + 1) * N], W[swapWith + int64_t(k + 1) * N]);
            }
            __syncthreads();
        }
        if (blockSize == 1)
        {
            const double d = W[k + int64_t(k) * N];
            for (int i = k + 1 + tid; i < N; i += BK_THREADS)
                F[i + int64_t(k) * N] = W[i + int64_t(k) * N] / d;
            if (tid == 0)
            {
                F[k + int64_t(k) * N] = d;
                fr.diag[k] = d;
                fr.sub[k] = 0.0;
            }
        }
        else
        {
            // LdltArithmetic's invertTwoByTwo: d11 = c/b, d22 = a/b, t = 1/(d11·d22 − 1), s = t/b.
            const double d0 = W[k + int64_t(k) * N], e = W[(k + 1) + int64_t(k) * N];
            const double d1 = W[(k + 1) + int64_t(k + 1) * N];
            const double d11 = d1 / e, d22 = d0 / e;
            const double t = 1.0 / (d11 * d22 - 1.0);
            const double s = t / e;
            for (int i = k + 2 + tid; i < N; i += BK_THREADS)
            {
                const double r0 = W[i + int64_t(k) * N], r1 = W[i + int64_t(k + 1) * N];
                F[i + int64_t(k) * N] = s * (d11 * r0 - r1);
                F[i + int64_t(k + 1) * N] = s * (d22 * r1 - r0);
            }
            if (tid == 0)
            {
                F[k + int64_t(k) * N] = d0;
                F[(k + 1) + int64_t(k) * N] = 0.0;
                F[(k + 1) + int64_t(k + 1) * N] = d1;
                fr.diag[k] = d0;
                fr.diag[k + 1] = d1;
                fr.sub[k] = e;
                fr.sub[k + 1] = 0.0;
            }
            ++twoByTwo;
        }
        __syncthreads();
        k += blockSize;
    }
    if (tid == 0)
        states[q] = PivotState{k, end, passStart, done, twoByTwo, k0, 0, 0};
}

// The value as an opaque register, in program order: the columns of a panel move down one by one, in place (left to the
// scheduler, old and new columns overlap and spill).
__device__ inline double pinned(double v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// A workgroup barrier for LDS alone: the stores of L and W in flight need not have landed.
__device__ inline void ldsBarrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The value a DPP control gives each lane (its own where the control has no source lane).
template <int CONTROL> __device__ inline double dppValue(double v)
{
    const long long bits = __builtin_bit_cast(long long, v);
    const int lo = int(bits), hi = int(bits >> 32);
    const unsigned l = unsigned(__builtin_amdgcn_update_dpp(lo, lo, CONTROL, 0xf, 0xf, false));
    const unsigned h = unsigned(__builtin_amdgcn_update_dpp(hi, hi, CONTROL, 0xf, 0xf, false));
    return __builtin_bit_cast(double, (static_cast<unsigned long long>(h) << 32) | l);
}

// The largest value of a wave, in its lane 63 (NaN ignored): shifts by 1, 2, 4 and 8 within rows of 16 lanes, then
// the rows' last lanes broadcast to the next ones.
__device__ inline double waveMax(double v)
{
    v = fmax(v, dppValue<0x111>(v));
    v = fmax(v, dppValue<0x112>(v));
    v = fmax(v, dppValue<0x114>(v));
    v = fmax(v, dppValue<0x118>(v));
    v = fmax(v, dppValue<0x142>(v));
    v = fmax(v, dppValue<0x143>(v));
    return v;
}

template <int WAVES> struct PanelShared
{
    // By the parity of the column: the waves' largest values, and the column's values in the panel's rows (its diagonal
    // first).
    double best[2][WAVES], row[2][PIVOT_PANEL];
    // Row imax of the panel, updated, and of the step's W; the waves' largest values of column imax, and its diagonal.
    double line[PIVOT_PANEL], wline[PIVOT_PANEL], rowBest[WAVES], corner;
    int at;
};

// A step of one front whose rows from the step's first column k0 on fit R per thread: the columns [k0, k0 + P) lie in
// registers, thread t holding rows k0 + t + THREADS·r, and are eliminated right-looking; each column done leaves the
// registers (its L and W stored) as the others move down by one, so the current column is always a[·][0]. A column
// costs one LDS barrier: the waves' maxima, the diagonal and W's row go through it together. Only the step's first
// column is interchanged or becomes a 2 × 2 pivot (in memory, where nothing of the step was done yet; the panel is
// then loaded again): a later column that needs it ends the step and is the next one's first.
//
// Bound by the latency of a column (the reduction, a division, the barrier): about 1.4 µs, where columns updated
// left-looking from L2 (64 to a step, pivotColumnsKernel) took 5 to 30 µs. 16 columns to a step: their product over
// the trailing candidates reads and writes those once per step, which HBM does beside nothing else (3,600 rows: 16 to
// 28 µs), so narrower steps pay there; wider ones do not fit the registers (R·P doubles: 128 VGPRs at R·P = 64). The
// 360 × 200 cylinder's factorisation took 328 ms before and 85 ms with these steps, launched without a wait between.
template <int THREADS, int R, int P>
__device__ void eliminatePanel(const PivotFront& fr, PivotState& st, PanelShared<THREADS / 64>& sh)
{
    constexpr int WAVES = THREADS / 64;
    double* F = fr.F;
    double* W = fr.W;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int64_t N = fr.N;
    const int n = fr.N, k0 = st.k;
    int k = k0, end = st.end;
    int forced = 0; // the first pivot is settled: 1 × 1 or 2 × 2
    double a[R][P];
    while (k < end)
    {
        const int pc = min(P, end - k0);
#pragma unroll
        for (int j = 0; j < P; ++j)
        {
            const double* column = F + (k0 + min(j, pc - 1)) * N;
#pragma unroll
            for (int r = 0; r < R; ++r)
                a[r][j] = column[unsigned(min(k0 + tid + THREADS * r, n - 1))];
        }
        if (forced == 2)
        {
            // LdltArithmetic's invertTwoByTwo: d11 = c/b, d22 = a/b, t = 1/(d11·d22 − 1), s = t/b.
            if (tid < pc)
            {
                sh.row[0][tid] = a[0][0]; // row k0 + tid
                sh.row[1][tid] = a[0][1];
            }
            __syncthreads();
            const double d0 = sh.row[0][0], e = sh.row[0][1], d1 = sh.row[1][1];
            const double d11 = d1 / e, d22 = d0 / e;
            const double t = 1.0 / (d11 * d22 - 1.0);
            const double s = t / e;
#pragma unroll
            for (int r = 0; r < R; ++r)
            {
                const int i = k0 + tid + THREADS * r;
                const double r0 = a[r][0], r1 = a[r][1];
                const double l0 = s * (d11 * r0 - r1), l1 = s * (d22 * r1 - r0);
                if (i > k0 + 1 && i < n)
                {
                    F[i + k0 * N] = l0;
                    F[i + (k0 + 1) * N] = l1;
                    W[i + k0 * N] = r0;
                    W[i + (k0 + 1) * N] = r1;
                }
#pragma unroll
                for (int j = 2; j < P; ++j)
                    a[r][j - 2] = pinned(a[r][j] - l0 * sh.row[0][j] - l1 * sh.row[1][j]);
            }
            if (tid == 0)
            {
                F[k0 + k0 * N] = d0;
                F[(k0 + 1) + k0 * N] = 0.0;
                F[(k0 + 1) + (k0 + 1) * N] = d1;
                fr.diag[k0] = d0;
                fr.diag[k0 + 1] = d1;
                fr.sub[k0] = e;
                fr.sub[k0 + 1] = 0.0;
            }
            ++st.twoByTwo;
            forced = 0;
            k += 2;
            __syncthreads(); // the rows are read
        }
        bool again = false; // the first column was interchanged, delayed or paired: load and go on
        while (k < k0 + pc)
        {
            const int parity = (k - k0) & 1, left = k0 + pc - k; // the columns still in the panel
            double m = 0.0;
#pragma unroll
            for (int r = 0; r < R; ++r)
            {
                const int i = k0 + tid + THREADS * r;
                if (i > k && i < n)
                    m = fmax(m, fabs(a[r][0]));
            }
            const int row = k0 + tid - k;
            if (row >= 0 && row < left) // the panel's rows: THREADS >= P
                sh.row[parity][row] = a[0][0];
            m = waveMax(m);
            if (lane == 63)
                sh.best[parity][wave] = m;
            ldsBarrier();
            double colmax = sh.best[parity][0];
#pragma unroll
            for (int w = 1; w < WAVES; ++w)
                colmax = fmax(colmax, sh.best[parity][w]);
            const double d = sh.row[parity][0], absakk = fabs(d);
            if (forced == 0 && absakk < BK_ALPHA * colmax)
            {
                // The first row of the largest value.
                __syncthreads();
                if (tid == 0)
                    sh.at = n;
                __syncthreads();
#pragma unroll
                for (int r = R - 1; r >= 0; --r)
                {
                    const int i = k0 + tid + THREADS * r;
                    if (i > k && i < n && fabs(a[r][0]) == colmax)
                        atomicMin(&sh.at, i);
                }
                __syncthreads();
                const int imax = sh.at;
                if (imax >= end)
                {
                    if (absakk < BK_DELAY * colmax)
                    {
                        // The partner is not a candidate and the diagonal is too small: delay the column.
                        if (k == k0)
                        {
                            --end;
                            if (k != end)
                                interchange<THREADS>(F, W, fr.perm, n, k, k, k, end);
                            again = true;
                        }
                        break;
                    }
                }
                else
                {
                    // Column imax, updated by the step's columns: its largest value besides its diagonal, and that.
                    if (tid < k - k0)
                        sh.wline[tid] = W[imax + (k0 + tid) * N];
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (k0 + tid + THREADS * r == imax)
                        {
#pragma unroll
                            for (int j = 0; j < P; ++j)
                                sh.line[j] = a[r][j];
                        }
                    __syncthreads();
                    const int at = imax - k;
                    double rowmax = 0.0;
#pragma unroll
                    for (int r = 0; r < R; ++r)
                    {
                        const int i = k0 + tid + THREADS * r;
                        if (i < k || i >= n)
                            continue;
                        double v;
                        if (i < imax && i < k + left)
                            v = sh.line[i - k];
                        else if (at < left)
                        {
                            v = a[r][0];
#pragma unroll
                            for (int j = 1; j < P; ++j)
                                v = j == at ? a[r][j] : v;
                        }
                        else
                        {
                            v = i >= imax ? F[i + imax * N] : F[imax + i * N];
                            constexpr int BATCH = 5; // loads in flight
                            for (int t0 = k0; t0 < k; t0 += BATCH)
                            {
                                double l[BATCH];
#pragma unroll
                                for (int t = 0; t < BATCH; ++t)
                                    l[t] = F[i + min(t0 + t, k - 1) * N];
#pragma unroll
                                for (int t = 0; t < BATCH; ++t)
                                    v = t0 + t < k ? v - pinned(l[t]) * sh.wline[t0 + t - k0] : v;
                            }
                        }
                        if (i == imax)
                            sh.corner = v;
                        else
                            rowmax = fmax(rowmax, fabs(v));
                    }
                    rowmax = waveMax(rowmax);
                    if (lane == 63)
                        sh.rowBest[wave] = rowmax;
                    __syncthreads();
                    rowmax = sh.rowBest[0];
#pragma unroll
                    for (int w = 1; w < WAVES; ++w)
                        rowmax = fmax(rowmax, sh.rowBest[w]);
                    if (!(absakk >= BK_ALPHA * colmax * (colmax / rowmax)))
                    {
                        if (k == k0)
                        {
                            forced = fabs(sh.corner) >= BK_ALPHA * rowmax ? 1 : 2;
                            __syncthreads(); // the tests are read
                            const int moved = k + forced - 1;
                            if (imax != moved)
                                interchange<THREADS>(F, W, fr.perm, n, k, k, moved, imax);
                            again = true;
                        }
                        break;
                    }
                }
            }
            const bool zero = d == 0.0 && colmax == 0.0; // a zero pivot: nothing to eliminate with it
            double l[R];
            double *Fk = F + k * N, *Wk = W + k * N;
#pragma unroll
            for (int r = 0; r < R; ++r)
            {
                const int i = k0 + tid + THREADS * r;
                l[r] = pinned(zero ? 0.0 : a[r][0] / d);
                if (i > k && i < n)
                {
                    Fk[unsigned(i)] = l[r];
                    Wk[unsigned(i)] = a[r][0];
                }
            }
#pragma unroll
            for (int j = 1; j < P; ++j)
            {
                const double w = sh.row[parity][j];
#pragma unroll
                for (int r = 0; r < R; ++r)
                    a[r][j - 1] = pinned(a[r][j] - l[r] * w);
            }
            if (tid == 0)
            {
                Fk[unsigned(k)] = d;
                fr.diag[k] = d;
                fr.sub[k] = 0.0;
            }
            forced = 0;
            ++k;
        }
        if (!again)
            break;
    }
    st.from = k0;
    st.k = k;
    st.end = end;
}

// One step of each front of the list, a workgroup per front, for fronts whose remaining rows fit the registers
// (PIVOT_SMALL_ROWS with 256 threads, PIVOT_LARGE_ROWS with 512).
template <int THREADS>
__global__ __launch_bounds__(THREADS) void pivotPanelKernel(const PivotFront* fronts, PivotState* states,
                                                            const int32_t* list)
{
    __shared__ PanelShared<THREADS / 64> sh;
    const int q = list[blockIdx.x];
    const PivotFront fr = fronts[q];
    PivotState st = states[q];
    st.from = st.k;
    if (!st.done && st.k == st.end)
    {
        if (st.end == fr.C || st.k == st.passStart)
            st.done = 1;
        else
        {
            st.passStart = st.k; // another pass over the delayed candidates
            st.end = fr.C;
        }
    }
    if (!st.done)
    {
        const int rows = fr.N - st.k;
        if (rows <= THREADS)
            eliminatePanel<THREADS, 1, PIVOT_PANEL>(fr, st, sh);
        else if (THREADS == 256 || rows <= 2 * THREADS)
            eliminatePanel<THREADS, 2, PIVOT_PANEL>(fr, st, sh);
        else if constexpr (THREADS == 512)
        {
            if (rows <= 4 * THREADS)
                eliminatePanel<THREADS, 4, PIVOT_PANEL>(fr, st, sh);
            else
                eliminatePanel<THREADS, 8, PIVOT_PANEL / 2>(fr, st, sh);
        }
        if (st.k == st.end && (st.end == fr.C || st.k == st.passStart))
            st.done = 1;
    }
    __syncthreads(); // every thread has read the state
    if (threadIdx.x == 0)
        states[q] = st;
}

// The trailing update of the last step: C −= L·Wᵀ over the step's columns [from, k), for the candidate columns and the
// rows from k on; item {front, row tile, column tile} of 64 × 64 at fixed positions of the front, four waves of
// 32 × 32 whose MFMA operands come straight from memory (K <= 17: nothing to reuse through LDS). Items whose columns
// are all eliminated do nothing.
__global__ __launch_bounds__(256) void pivotTrailingKernel(const PivotFront* fronts, const PivotState* states,
                                                           const int4* items)
{
    const int4 item = items[blockIdx.x];
    const PivotState st = states[item.x];
    const PivotFront fr = fronts[item.x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row0 = 64 * item.y + 32 * (wave >> 1), col0 = 64 * item.z + 32 * (wave & 1);
    const int from = st.from, k = st.k, n = fr.N;
    if (from == k || col0 + 32 <= k || col0 >= fr.C || row0 >= n || row0 + 32 <= max(k, col0))
        return;
    const int64_t N = n;
    const int lr = lane & 15, lq = lane >> 4;
    double4_t acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int i = min(row0 + 16 * x + lq + 4 * v, n - 1), j = min(col0 + 16 * y + lr, n - 1);
                acc[x][y][v] = fr.F[i + j * N];
            }
    for (int t0 = from; t0 < k; t0 += 4)
    {
        const int t = min(t0 + lq, k - 1);
        double av[2], bv[2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
        {
            av[x] = fr.F[min(row0 + 16 * x + lr, n - 1) + t * N];
            bv[x] = fr.W[min(col0 + 16 * x + lr, n - 1) + t * N];
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
        {
            av[x] = t0 + lq < k ? -av[x] : 0.0;
            bv[x] = t0 + lq < k ? bv[x] : 0.0;
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
                acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[x], bv[y], acc[x][y], 0, 0, 0);
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int i = row0 + 16 * x + lq + 4 * v, j = col0 + 16 * y + lr;
                if (i < n && j < fr.C && i >= j && j >= k)
                    fr.F[i + j * N] = acc[x][y][v];
            }
}

// The matrix entries of each front's own columns, at their positions (rows past the own columns move down by the
// delayed count). The front is zero before.
__global__ __launch_bounds__(256) void pivotMatrixKernel(DeviceMatrix a, const PivotFront* fronts)
{
    const PivotFront fr = fronts[blockIdx.x];
    const int64_t kb = a.offsets[fr.first], ke = a.offsets[fr.first + fr.c];
    for (int64_t q = kb + threadIdx.x; q < ke; q += blockDim.x)
    {
        const int pos = a.position[q], j = a.column[q];
        const int at = pos < fr.c ? pos : pos + fr.d;
        fr.F[at + int64_t(j) * fr.N] += a.values[q];
    }
}

// The extend-add of one child's update matrix (columns [j0, j1) of it) into its parent's front: entry (i, j), i >= j,
// goes to the parent's positions (map[i], map[j]) ordered into the lower triangle. A child's positions are distinct,
// so no two threads meet; children of one parent go in separate launches, in order.
__global__ __launch_bounds__(256) void pivotExtendAddKernel(const ExtendItem* items)
{
    const ExtendItem it = items[blockIdx.x];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int j = it.j0 + wave; j < it.j1; j += 4)
    {
        const int pj = it.map[j];
        for (int i = j + lane; i < it.M; i += 64)
        {
            const int pi = it.map[i];
            const int r = max(pi, pj), c = min(pi, pj);
            it.dst[r + int64_t(c) * it.ldd] += it.src[i + int64_t(j) * it.lds];
        }
    }
}

// Contiguous copies (the eliminated columns of the fronts into the panels).
__global__ __launch_bounds__(256) void copyRangesKernel(const CopyRange* ranges)
{
    const CopyRange r = ranges[blockIdx.x];
    for (int64_t q = threadIdx.x; q < r.count; q += blockDim.x)
        r.dst[q] = r.src[q];
}

// The inverse of a 64-column diagonal block (s, J) of a unit lower triangle L_FF (the strictly lower values of the
// panel; the diagonal taken as 1): kb × kb column-major at linvOff[s] + 64·64·J, leading dimension kb. Column j of
// the inverse by forward substitution on one lane each.
__global__ __launch_bounds__(64) void unitBlockInverseKernel(DevicePlan p, const double* panels, double* linv,
                                                             const int2* items)
{
    __shared__ double Ls[PANEL_BLOCK][PANEL_BLOCK + 1];
    __shared__ double Xs[PANEL_BLOCK][PANEL_BLOCK + 1];
    const int2 item = items[blockIdx.x];
    const int s = item.x, q0 = item.y * PANEL_BLOCK;
    const int c = p.ncol[s], n = c + p.nrow[s];
    const int kb = min(PANEL_BLOCK, c - q0);
    const double* L = panels + p.panelOff[s] + q0 + int64_t(q0) * n;
    const int lane = threadIdx.x;
    for (int j = 0; j < kb; ++j)
        if (lane < kb)
            Ls[lane][j] = lane > j ? L[lane + int64_t(j) * n] : 0.0;
    __syncthreads();
    if (lane < kb)
    {
        const int j = lane;
        for (int i = 0; i < kb; ++i)
            Xs[i][j] = i == j ? 1.0 : 0.0;
        for (int i = j + 1; i < kb; ++i)
        {
            double x = 0.0;
            for (int t = j; t < i; ++t)
                x -= Ls[i][t] * Xs[t][j];
            Xs[i][j] = x;
        }
    }
    __syncthreads();
    double* out = linv + p.linvOff[s] + int64_t(q0) * PANEL_BLOCK;
    for (int j = 0; j < kb; ++j)
        if (lane < kb)
            out[lane + j * kb] = Xs[lane][j];
}

// X ← D⁻¹·X for a block diagonal D (X row-major n × k): 1 × 1 pivots divide; a 2 × 2 block (sub[i] != 0, rows i and
// i + 1) is solved by LdltArithmetic's inverse, x0 = s·(d11·b0 − b1), x1 = s·(d22·b1 − b0).
__global__ __launch_bounds__(256) void blockDiagonalSolveKernel(double* X, const double* d, const double* sub,
                                                                int64_t n, int k)
{
    const int h = threadIdx.x & 15;
    const int64_t i = blockIdx.x * int64_t(blockDim.x >> 4) + (threadIdx.x >> 4);
    if (h >= k || i >= n)
        return;
    if (i > 0 && sub[i - 1] != 0.0)
        return; // the second row of a block, solved with the first
    if (sub[i] != 0.0 && i + 1 < n)
    {
        const double a = d[i], e = sub[i], c = d[i + 1];
        const double d11 = c / e, d22 = a / e;
        const double t = 1.0 / (d11 * d22 - 1.0);
        const double s = t / e;
        const double b0 = X[i * k + h], b1 = X[(i + 1) * k + h];
        X[i * k + h] = s * (d11 * b0 - b1);
        X[(i + 1) * k + h] = s * (d22 * b1 - b0);
        return;
    }
    X[i * k + h] = X[i * k + h] / d[i];
}

// dst[i] = src[perm[i]] (gather) or dst[perm[i]] = src[i] (scatter), rows of k values.
__global__ __launch_bounds__(256) void permuteRowsKernel(const double* src, double* dst, const int32_t* perm,
                                                         int64_t n, int k, int scatter)
{
    const int h = threadIdx.x & 15;
    const int64_t i = blockIdx.x * int64_t(blockDim.x >> 4) + (threadIdx.x >> 4);
    if (h >= k || i >= n)
        return;
    const int64_t at = perm[i];
    if (scatter)
        dst[at * k + h] = src[i * k + h];
    else
        dst[i * k + h] = src[at * k + h];
}

int rowGroups(int64_t n)
{
    return static_cast<int>((n + 15) / 16);
}

} // namespace

hipError_t launchPivotStep(int kind, const PivotFront* fronts, PivotState* states, const int32_t* list, int count,
                           hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    if (kind == PIVOT_SMALL)
        hipLaunchKernelGGL(pivotPanelKernel<256>, dim3(count), dim3(256), 0, stream, fronts, states, list);
    else if (kind == PIVOT_LARGE)
        hipLaunchKernelGGL(pivotPanelKernel<512>, dim3(count), dim3(512), 0, stream, fronts, states, list);
    else
        hipLaunchKernelGGL(pivotColumnsKernel, dim3(count), dim3(BK_THREADS), 0, stream, fronts, states, list,
                           PIVOT_PANEL / 2);
    return hipGetLastError();
}

hipError_t launchPivotTrailing(const PivotFront* fronts, const PivotState* states, const int4* items, int count,
                               hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    hipLaunchKernelGGL(pivotTrailingKernel, dim3(count), dim3(256), 0, stream, fronts, states, items);
    return hipGetLastError();
}

hipError_t launchPivotMatrix(const DeviceMatrix& a, const PivotFront* fronts, int count, hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    hipLaunchKernelGGL(pivotMatrixKernel, dim3(count), dim3(256), 0, stream, a, fronts);
    return hipGetLastError();
}

hipError_t launchPivotExtendAdd(const ExtendItem* items, int count, hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    hipLaunchKernelGGL(pivotExtendAddKernel, dim3(count), dim3(256), 0, stream, items);
    return hipGetLastError();
}

hipError_t launchCopyRanges(const CopyRange* ranges, int count, hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    hipLaunchKernelGGL(copyRangesKernel, dim3(count), dim3(256), 0, stream, ranges);
    return hipGetLastError();
}

hipError_t launchUnitBlockInverses(const DevicePlan& p, const double* panels, double* linv, const int2* items,
                                   int count, hipStream_t stream)
{
    if (count == 0)
        return hipSuccess;
    hipLaunchKernelGGL(unitBlockInverseKernel, dim3(count), dim3(64), 0, stream, p, panels, linv, items);
    return hipGetLastError();
}

hipError_t launchBlockDiagonalSolve(double* X, const double* d, const double* sub, int64_t n, int k,
                                    hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    hipLaunchKernelGGL(blockDiagonalSolveKernel, dim3(rowGroups(n)), dim3(256), 0, stream, X, d, sub, n, k);
    return hipGetLastError();
}

hipError_t launchPermuteRows(const double* src, double* dst, const int32_t* perm, int64_t n, int k, bool scatter,
                             hipStream_t stream)
{
    if (n == 0)
        return hipSuccess;
    hipLaunchKernelGGL(permuteRowsKernel, dim3(rowGroups(n)), dim3(256), 0, stream, src, dst, perm, n, k,
                       scatter ? 1 : 0);
    return hipGetLastError();
}

} // namespace oosg
