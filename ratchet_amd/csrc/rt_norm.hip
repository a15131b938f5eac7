// LayerNorm, RMSNorm (one wave64 per row, row held in registers, 16-byte loads, butterfly reductions) and GroupNorm
// (groups of up to 192 or 256 KiB in the registers of a block, one launch; larger ones in slices, statistics + apply, two launches).
//
// Arithmetic contract for LayerNorm / RMSNorm = crates/ratchet-core/src/cpu/norm.rs:91-147,185-213, in the element type T
// with one rounding per operation:
//     mu   = sum(x) / T(N)                 (sum::<T>: f32 accumulation; for 16-bit T rounded to T once)
//     x2   = sum(x*x) / T(N)               (each square rounded to T first)
//     var  = x2 - mu*mu                    (E[x^2] - mu^2, not a two-pass variance)
//     r    = T(1) / sqrt(var + T(eps))
//     y    = ((x - mu) * r) * scale + bias
// f32 rows: one wave64 per row, the row stays in registers, the additions form a butterfly tree instead of the
//   reference's sequential fold; that changes the sums by float rounding only (far inside the 1e-5 bar).
// 16-bit rows: the two sums are rounded to the 16-bit type before they are used (sum(x*x) ~ N has an ulp of 1-2 there),
//   so a different f32 summation order can flip that rounding and move a whole row by an ulp of r, more than 1e-3
//   allows.  These kernels therefore replay the reference's order exactly: tiles of x and T(x*x) are staged through LDS
//   as f32 and one lane per (row, sum) walks its row left to right with v_add_f32.  The walk is latency bound
//   (one dependent add per element), so many small row groups run side by side.  Where it is faster a wave per row finds what
//   the ordered sum rounds to without walking it (rt_norm_row.hip).
// GroupNorm follows torch.nn.functional.group_norm, the ground truth of the reference's own test
// (ops/norm/groupnorm.rs:24-31): sums in f32 inside a thread (a slice), joined in double, f32 arithmetic, one final rounding.
#include <type_traits>

#include "rt_arith.h"
#include "rt_internal.h"
#include "rt_norm.h"

namespace {

constexpr int WAVE = 64;
constexpr int BLOCK = 256;
constexpr int WAVES = BLOCK / WAVE;

// Partial statistics for rt_group_norm_static, the entry point that allocates nothing: a fixed array in the code object,
// one copy per GPU.  In host code the array's name is only a stand-in; rt_norm_device_init asks the runtime where the
// current device's copy lies and every launch is given that pointer.
constexpr size_t GN_STATIC_SCRATCH_BYTES = 256 * 1024;
static __device__ __align__(256) unsigned char gn_static_scratch[GN_STATIC_SCRATCH_BYTES];
constexpr int NORM_WIDE_BLOCK = 1024;                   // threads per row for f32 rows that do not fit 256 threads' registers

// x and y 16-byte aligned, at most LANES * NV vectors per row.  Rows of whole vectors (scale and bias 16-byte aligned as
// well), or SPAN: rows of any length over the aligned vectors that cover them.  A row then starts `shift` elements into
// its first vector; span elements outside the row belong to the neighbouring rows, stay out of the sums and are not
// written (the row's two ragged vectors are stored element by element), and scale / bias are read by column.  An
// aligned vector that holds one byte of the tensor lies in a mapped page, so the loads are safe at the tensor's ends too.
template <typename T, int NV, int KIND, int LANES, bool SPAN>
__global__ void __launch_bounds__(LANES > BLOCK ? LANES : BLOCK) norm_wave_kernel(const T* x, const T* __restrict__ scale,
                                                                                  const T* __restrict__ bias, T* y, uint64_t rows,
                                                                                  uint32_t cols, float eps) {
    constexpr int VE = 16 / sizeof(T);
    constexpr int THREADS = LANES > BLOCK ? LANES : BLOCK;   // rows beyond 2048 vectors: one 1024-thread block per row
    const uint64_t row = (uint64_t)blockIdx.x * (THREADS / LANES) + (threadIdx.x / LANES);
    if (row >= rows) return;
    const int lane = threadIdx.x & (LANES - 1);
    const uint64_t first = row * cols;
    const uint32_t shift = SPAN ? (uint32_t)(first & (VE - 1)) : 0;
    const uint32_t nvec = SPAN ? (shift + cols + VE - 1) / VE : cols / VE;
    const v4u* xr = reinterpret_cast<const v4u*>(x) + first / VE;
    v4u* yr = reinterpret_cast<v4u*>(y) + first / VE;
    auto inside = [&](uint32_t i, int q) -> bool { return !SPAN || i * VE + (uint32_t)q - shift < cols; };
    Vec16<T> v[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = lane + k * LANES;
        if (i < nvec) v[k].u = ld_stream(xr + i);
    }
    float sx = 0.0f, sq = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; k++)
        if (lane + k * LANES < nvec)
#pragma unroll
            for (int q = 0; q < VE; q++)
                if (inside(lane + k * LANES, q)) {
                    const T e = v[k].e[q];
                    if (KIND == NORM_LAYER) sx += Ar<T>::widen(e);
                    sq += Ar<T>::widen(Ar<T>::mul(e, e));
                }
    if (KIND == NORM_LAYER) sx = row_sum<LANES>(sx);
    sq = row_sum<LANES>(sq);
    const RowStats<T> st = finish_stats<T, KIND>(sx, sq, cols, eps);
    const v4u* sv = reinterpret_cast<const v4u*>(scale);
    const v4u* bv = reinterpret_cast<const v4u*>(bias);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = lane + k * LANES;
        if (i < nvec) {
            Vec16<T> s, b, o;
            if (!SPAN) {
                s.u = sv[i];
                if (KIND == NORM_LAYER && bias) b.u = bv[i];
#pragma unroll
                for (int q = 0; q < VE; q++) o.e[q] = norm_one<T, KIND>(v[k].e[q], st, s.e[q], b.e[q], bias != nullptr);
                st_stream(yr + i, o.u);
            } else if (inside(i, 0) && inside(i, VE - 1)) {
                // a vector inside the row: its scale / bias elements are 16 contiguous bytes at element alignment
                const uint32_t c0 = i * VE - shift;
                __builtin_memcpy(&s.u, scale + c0, 16);
                if (KIND == NORM_LAYER && bias) __builtin_memcpy(&b.u, bias + c0, 16);
#pragma unroll
                for (int q = 0; q < VE; q++) o.e[q] = norm_one<T, KIND>(v[k].e[q], st, s.e[q], b.e[q], bias != nullptr);
                st_stream(yr + i, o.u);
            } else {
                T* yrow = y + first;
#pragma unroll
                for (int q = 0; q < VE; q++) {
                    const uint32_t c = i * VE + (uint32_t)q - shift;
                    if (c < cols) {
                        const T bq = (KIND == NORM_LAYER && bias) ? bias[c] : Ar<T>::conv(0.0f);
                        yrow[c] = norm_one<T, KIND>(v[k].e[q], st, scale[c], bq, bias != nullptr);
                    }
                }
            }
        }
    }
}

// any cols / alignment: one block per row, scalar accesses, the row is re-read from cache for the second pass
template <typename T, int KIND>
__global__ void __launch_bounds__(BLOCK) norm_generic_kernel(const T* __restrict__ x, const T* __restrict__ scale,
                                                             const T* __restrict__ bias, T* __restrict__ y, uint64_t rows, uint32_t cols,
                                                             float eps) {
    __shared__ float red[2][WAVES];
    const uint64_t row = blockIdx.x;
    const T* xr = x + row * cols;
    T* yr = y + row * cols;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    float sx = 0.0f, sq = 0.0f;
    for (uint32_t j = threadIdx.x; j < cols; j += BLOCK) {
        const T e = xr[j];
        sx += Ar<T>::widen(e);
        sq += Ar<T>::widen(Ar<T>::mul(e, e));
    }
    sx = wave_sum(sx);
    sq = wave_sum(sq);
    if (lane == 0) { red[0][wave] = sx; red[1][wave] = sq; }
    __syncthreads();
    sx = red[0][0]; sq = red[1][0];
    for (int w = 1; w < WAVES; w++) { sx += red[0][w]; sq += red[1][w]; }
    const RowStats<T> st = finish_stats<T, KIND>(sx, sq, cols, eps);
    for (uint32_t j = threadIdx.x; j < cols; j += BLOCK) {
        const T b = (KIND == NORM_LAYER && bias) ? bias[j] : Ar<T>::conv(0.0f);
        yr[j] = norm_one<T, KIND>(xr[j], st, scale[j], b, bias != nullptr);
    }
}

// ------------------------------------------------------------------------------------------------------------------
// The caller pattern of ratchet-nn (src/norm.rs:35-44, 61-70): x.full().layer_norm(w, b, eps).cast(src_dt) on a
// 16-bit x with f32 weights, in one pass: the row is widened into registers, the f32 norm arithmetic above is applied
// (butterfly sums) and the result is rounded once.  4 bytes of traffic per element instead of the 16 of the three
// separate ops, and no sequential chain: the f32 sums need no replay because the parity bar after the cast is the
// 16-bit one.
// ------------------------------------------------------------------------------------------------------------------
template <typename T, int NV, int KIND, int LANES>
__global__ void __launch_bounds__(BLOCK) norm_via32_wave_kernel(const T* __restrict__ x, const float* __restrict__ scale,
                                                                const float* __restrict__ bias, T* __restrict__ y, uint64_t rows,
                                                                uint32_t cols, float eps) {
    const uint64_t row = (uint64_t)blockIdx.x * (BLOCK / LANES) + (threadIdx.x / LANES);
    if (row >= rows) return;
    const int lane = threadIdx.x & (LANES - 1);
    const uint32_t nvec = cols / 8;
    const v4u* xr = reinterpret_cast<const v4u*>(x + row * cols);
    v4u* yr = reinterpret_cast<v4u*>(y + row * cols);
    Vec16<T> v[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = lane + k * LANES;
        if (i < nvec) v[k].u = ld_stream(xr + i);
    }
    float sx = 0.0f, sq = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; k++)
        if (lane + k * LANES < nvec)
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const float e = Ar<T>::widen(v[k].e[q]);
                if (KIND == NORM_LAYER) sx += e;
                sq += e * e;
            }
    if (KIND == NORM_LAYER) sx = row_sum<LANES>(sx);
    sq = row_sum<LANES>(sq);
    const RowStats<float> st = finish_stats<float, KIND>(sx, sq, cols, eps);
    const float4* sv = reinterpret_cast<const float4*>(scale);
    const float4* bv = reinterpret_cast<const float4*>(bias);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = lane + k * LANES;
        if (i < nvec) {
            float s[8], b[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            *reinterpret_cast<float4*>(s) = sv[2 * i];
            *reinterpret_cast<float4*>(s + 4) = sv[2 * i + 1];
            if (KIND == NORM_LAYER && bias) {
                *reinterpret_cast<float4*>(b) = bv[2 * i];
                *reinterpret_cast<float4*>(b + 4) = bv[2 * i + 1];
            }
            Vec16<T> o;
#pragma unroll
            for (int q = 0; q < 8; q++)
                o.e[q] = Ar<T>::conv(norm_one<float, KIND>(Ar<T>::widen(v[k].e[q]), st, s[q], b[q], bias != nullptr));
            st_stream(yr + i, o.u);
        }
    }
}

// RW rows per wave (or per block, LANES == BLOCK): the f32 weights are twice the bytes of a 16-bit row (four times with a
// bias), and every row fetches them again, behind its reduction, where only the other waves hide the wait
// ([16384,4096] LayerNorm 52.8 us; without the weight loads 46.1 us; a copy of the same bytes 42.9 us).  With RW rows in
// registers the weights of a vector are loaded once and applied RW times.  The launcher says where that pays.
template <typename T, int NV, int KIND, int LANES, int RW>
__global__ void __launch_bounds__(BLOCK) norm_via32_rows_kernel(const T* __restrict__ x, const float* __restrict__ scale,
                                                                const float* __restrict__ bias, T* __restrict__ y, uint64_t rows,
                                                                uint32_t cols, float eps) {
    const uint64_t row0 = ((uint64_t)blockIdx.x * (BLOCK / LANES) + (threadIdx.x / LANES)) * RW;
    if (row0 >= rows) return;
    const int lane = threadIdx.x & (LANES - 1);
    const uint32_t nvec = cols / 8;
    Vec16<T> v[RW][NV];
#pragma unroll
    for (int r = 0; r < RW; r++) {
        // a row past the end reads the last row once more (its result is not stored): no branch around the loads
        const uint64_t row = row0 + r < rows ? row0 + r : rows - 1;
        const v4u* xr = reinterpret_cast<const v4u*>(x + row * cols);
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const uint32_t i = lane + k * LANES;
            if (i < nvec) v[r][k].u = ld_stream(xr + i);
        }
    }
    RowStats<float> st[RW];
#pragma unroll
    for (int r = 0; r < RW; r++) {
        float sx = 0.0f, sq = 0.0f;
#pragma unroll
        for (int k = 0; k < NV; k++)
            if (lane + k * LANES < nvec)
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const float e = Ar<T>::widen(v[r][k].e[q]);
                    if (KIND == NORM_LAYER) sx += e;
                    sq += e * e;
                }
        if (KIND == NORM_LAYER) sx = row_sum<LANES>(sx);
        sq = row_sum<LANES>(sq);
        st[r] = finish_stats<float, KIND>(sx, sq, cols, eps);
    }
    const float4* sv = reinterpret_cast<const float4*>(scale);
    const float4* bv = reinterpret_cast<const float4*>(bias);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = lane + k * LANES;
        if (i < nvec) {
            float s[8], b[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            *reinterpret_cast<float4*>(s) = sv[2 * i];
            *reinterpret_cast<float4*>(s + 4) = sv[2 * i + 1];
            if (KIND == NORM_LAYER && bias) {
                *reinterpret_cast<float4*>(b) = bv[2 * i];
                *reinterpret_cast<float4*>(b + 4) = bv[2 * i + 1];
            }
#pragma unroll
            for (int r = 0; r < RW; r++) {
                if (row0 + r >= rows) break;
                Vec16<T> o;
#pragma unroll
                for (int q = 0; q < 8; q++)
                    o.e[q] = Ar<T>::conv(norm_one<float, KIND>(Ar<T>::widen(v[r][k].e[q]), st[r], s[q], b[q], bias != nullptr));
                st_stream(reinterpret_cast<v4u*>(y + (row0 + r) * cols) + i, o.u);
            }
        }
    }
}

// any cols / alignment: one block per row, scalar accesses, the row is re-read from cache for the second pass
template <typename T, int KIND>
__global__ void __launch_bounds__(BLOCK) norm_via32_generic_kernel(const T* __restrict__ x, const float* __restrict__ scale,
                                                                   const float* __restrict__ bias, T* __restrict__ y, uint64_t rows,
                                                                   uint32_t cols, float eps) {
    __shared__ float red[2][WAVES];
    const uint64_t row = blockIdx.x;
    const T* xr = x + row * cols;
    T* yr = y + row * cols;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    float sx = 0.0f, sq = 0.0f;
    for (uint32_t j = threadIdx.x; j < cols; j += BLOCK) {
        const float e = Ar<T>::widen(xr[j]);
        sx += e;
        sq += e * e;
    }
    sx = wave_sum(sx);
    sq = wave_sum(sq);
    if (lane == 0) { red[0][wave] = sx; red[1][wave] = sq; }
    __syncthreads();
    sx = red[0][0]; sq = red[1][0];
    for (int w = 1; w < WAVES; w++) { sx += red[0][w]; sq += red[1][w]; }
    const RowStats<float> st = finish_stats<float, KIND>(sx, sq, cols, eps);
    for (uint32_t j = threadIdx.x; j < cols; j += BLOCK) {
        const float b = (KIND == NORM_LAYER && bias) ? bias[j] : 0.0f;
        yr[j] = Ar<T>::conv(norm_one<float, KIND>(Ar<T>::widen(xr[j]), st, scale[j], b, bias != nullptr));
    }
}

// ------------------------------------------------------------------------------------------------------------------
// 16-bit LayerNorm / RMSNorm with the reference's sequential f32 accumulation.
// A block owns RB consecutive rows.  Pass A: per column tile, all threads load elements, widen x and T(x*x) to f32 and park
// them in LDS; lanes [0, RB) then add the squares of "their" row left to right, lanes [RB, 2RB) the values
// (LayerNorm only).  Pass B re-reads x (from cache: the block touched it moments ago), normalises and stores.
// ------------------------------------------------------------------------------------------------------------------
template <typename T, int RB, int KIND>
__global__ void __launch_bounds__(BLOCK) norm_seq16_kernel(const T* __restrict__ x, const T* __restrict__ scale,
                                                           const T* __restrict__ bias, T* __restrict__ y, uint64_t rows, uint32_t cols,
                                                           float eps) {
    constexpr int TC = 128;
    constexpr int PAD = 4;
    constexpr int NSUM = (KIND == NORM_LAYER) ? 2 : 1;
    __shared__ __attribute__((aligned(16))) float tile[NSUM][RB][TC + PAD];      // [0] = squares, [1] = values
    __shared__ float sums[NSUM][RB];
    __shared__ T s_mu[RB], s_r[RB];
    const uint64_t row0 = (uint64_t)blockIdx.x * RB;
    const uint32_t nrows = (rows - row0 < (uint64_t)RB) ? (uint32_t)(rows - row0) : (uint32_t)RB;
    const uint32_t wrow = threadIdx.x % RB, wsum = threadIdx.x / RB;                // walker role of this thread
    const bool walker = (threadIdx.x < NSUM * RB) && (wrow < nrows);
    float run = 0.0f;

    for (uint32_t c0 = 0; c0 < cols; c0 += TC) {
        const uint32_t ncol = (cols - c0 < (uint32_t)TC) ? cols - c0 : (uint32_t)TC;
        for (uint32_t idx = threadIdx.x; idx < (uint32_t)RB * TC; idx += BLOCK) {
            const uint32_t r = idx / TC, col = idx % TC;
            if (r < nrows && col < ncol) {
                const T e = x[(row0 + r) * cols + c0 + col];
                tile[0][r][col] = Ar<T>::widen(Ar<T>::mul(e, e));
                if (KIND == NORM_LAYER) tile[NSUM - 1][r][col] = Ar<T>::widen(e);
            }
        }
        __syncthreads();
        if (walker) {
            const float* trow = tile[wsum][wrow];
            uint32_t j = 0;
            for (; j + 4 <= ncol; j += 4) {
                const float4 t = *reinterpret_cast<const float4*>(trow + j);
                run += t.x;
                run += t.y;
                run += t.z;
                run += t.w;
            }
            for (; j < ncol; j++) run += trow[j];
        }
        __syncthreads();
    }
    if (walker) sums[wsum][wrow] = run;
    __syncthreads();
    if (threadIdx.x < nrows) {
        const RowStats<T> st = finish_stats<T, KIND>(KIND == NORM_LAYER ? sums[NSUM - 1][threadIdx.x] : 0.0f, sums[0][threadIdx.x],
                                                     cols, eps);
        s_mu[threadIdx.x] = st.mu;
        s_r[threadIdx.x] = st.r;
    }
    __syncthreads();

    for (uint32_t r = 0; r < nrows; r++) {
        RowStats<T> st;
        st.mu = s_mu[r];
        st.r = s_r[r];
        const T* src = x + (row0 + r) * cols;
        T* dst = y + (row0 + r) * cols;
        for (uint32_t c = threadIdx.x; c < cols; c += BLOCK) {
            const T b = (KIND == NORM_LAYER && bias) ? bias[c] : Ar<T>::conv(0.0f);
            dst[c] = norm_one<T, KIND>(src[c], st, scale[c], b, bias != nullptr);
        }
    }
}

// Pipelined form of the kernel above for the common case (cols % 8 == 0, 16-byte aligned operands).
// 8 rows per 320-thread block, 256-column tiles.  Wave 0 does nothing but walk (8 lanes for RMSNorm, 16 for LayerNorm)
// and raises its issue priority; the four loader waves fetch one 16-byte vector per thread per tile two tiles ahead,
// widen x and T(x*x) to f32 and park them in double-buffered LDS tiles; one barrier per tile.  The kernel runs at the
// speed of the walk.  A dependent v_add_f32 takes 4.9 cycles (2.0 ns) on this chip, but the walker also has to issue its
// own LDS reads, one per four values of an f32 tile, which brings a column to about 3 ns.  For f16 the tiles therefore
// hold the 16-bit values themselves (x, and T(x*x), which is an f16 value too): one LDS read per eight values, and the
// chain adds them with v_fma_mix_f32 (1.0 * f16 operand + running f32 sum: the same sum, the widening is part of the
// instruction).  bf16 has no such instruction and keeps the f32 tiles.
// KEEP (launches whose blocks are all resident at once, rows of at most NP_KEEP_MAX_COLS columns): the walk of every row
// of the tensor then ends at the same moment and nothing can hide what comes after it, so the output pass must be
// nothing but stores: each loader thread also parks the raw vectors it loaded in dynamic LDS, scale and bias are staged
// there once at the start, and after the statistics the block reads LDS, normalises and streams the result out,
// instead of fetching x a second time through a loop of dependent load / store pairs.
constexpr int NP_BLOCK = 320;
constexpr uint32_t NP_KEEP_MAX_COLS = 4096;
constexpr size_t NP_KEEP_BYTES_PER_TILE = 256 * 16 + 2 * 32 * 16;   // the block's x vectors, one scale and one bias vector per column group
// run += the 32 f16 values packed in four vectors, left to right: each add is 1.0 * widen(f16) + run in one instruction
// with one rounding, which is the f32 sum of the widened values.  One asm statement for the whole run of adds: between
// separate statements the compiler, which cannot see into them, puts wait states that cost more than the adds.
#define NP_MIX_LO(N) "v_fma_mix_f32 %0, %" #N ", %17, %0 op_sel_hi:[1,0,0]\n"
#define NP_MIX_HI(N) "v_fma_mix_f32 %0, %" #N ", %17, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n"
#define NP_MIX(N) NP_MIX_LO(N) NP_MIX_HI(N)
__device__ __forceinline__ void np_add_f16x32(float& run, const v4u& a, const v4u& b, const v4u& c, const v4u& d) {
    const float one = 1.0f;
    asm(NP_MIX(1) NP_MIX(2) NP_MIX(3) NP_MIX(4) NP_MIX(5) NP_MIX(6) NP_MIX(7) NP_MIX(8) NP_MIX(9) NP_MIX(10) NP_MIX(11) NP_MIX(12)
        NP_MIX(13) NP_MIX(14) NP_MIX(15) NP_MIX(16)
        : "+v"(run)
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]),
          "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]), "s"(one));
}
#undef NP_MIX
#undef NP_MIX_HI
#undef NP_MIX_LO
template <typename T, int KIND, bool KEEP>
__global__ void __launch_bounds__(NP_BLOCK) norm_pipe16_kernel(const T* __restrict__ x, const T* __restrict__ scale,
                                                               const T* __restrict__ bias, T* __restrict__ y, uint64_t rows, uint32_t cols,
                                                               float eps) {
    constexpr int RB = 8, TC = 256, PAD = 4, PAD16 = 8;
    constexpr int NSUM = (KIND == NORM_LAYER) ? 2 : 1;
    constexpr bool H16 = std::is_same<T, half_t>::value;                         // 16-bit tiles and the fma_mix chain
    // [.][0] = squares, [.][1] = values: f32, or the f16 bit patterns
    __shared__ __attribute__((aligned(16))) unsigned char tile_raw[H16 ? 2 * NSUM * RB * (TC + PAD16) * 2 : 2 * NSUM * RB * (TC + PAD) * 4];
    float (*tile)[NSUM][RB][TC + PAD] = reinterpret_cast<float (*)[NSUM][RB][TC + PAD]>(tile_raw);
    uint16_t (*tile16)[NSUM][RB][TC + PAD16] = reinterpret_cast<uint16_t (*)[NSUM][RB][TC + PAD16]>(tile_raw);
    __shared__ float sums[NSUM][RB];
    __shared__ T s_mu[RB], s_r[RB];
    extern __shared__ __attribute__((aligned(16))) v4u np_keep[];               // KEEP: [ntiles][256] x, [ntiles][32] scale, [ntiles][32] bias
    const uint64_t row0 = (uint64_t)blockIdx.x * RB;
    const uint32_t nrows = (rows - row0 < (uint64_t)RB) ? (uint32_t)(rows - row0) : (uint32_t)RB;
    const uint32_t ntiles = (cols + TC - 1) / TC;

    if (threadIdx.x < 64) {
        // ---------------------------------------------------------------- wave 0: the sequential sums
        __builtin_amdgcn_s_setprio(3);
        const uint32_t wrow = threadIdx.x % RB, wsum = (threadIdx.x / RB) % NSUM;   // lanes beyond NSUM*RB shadow and never publish
        const bool publish = (threadIdx.x < NSUM * RB) && (wrow < nrows);
        float run = 0.0f;
        if constexpr (H16) {
            // The barrier that says "tile t + 1 is in LDS" is taken before the last 32 adds of tile t, whose operands are in
            // registers by then (the loaders may overwrite tile t after it): the first LDS reads of the next tile are in
            // flight during those adds, so the chain never waits for LDS at a tile's start.
            __syncthreads();                                                    // tile 0 is in LDS
            v4u cur[4], nxt[4];
            {
                const v4u* first = reinterpret_cast<const v4u*>(tile16[0][wsum][wrow]);
#pragma unroll
                for (int k = 0; k < 4; k++) cur[k] = first[k];
            }
            for (uint32_t t = 0; t < ntiles; t++) {
                const v4u* trow16 = reinterpret_cast<const v4u*>(tile16[t & 1][wsum][wrow]);
                const v4u* trow16n = reinterpret_cast<const v4u*>(tile16[(t + 1) & 1][wsum][wrow]);
#pragma unroll
                for (int c = 0; c < TC / 32; c++) {
                    if (c + 1 < TC / 32) {
#pragma unroll
                        for (int k = 0; k < 4; k++) nxt[k] = trow16[(c + 1) * 4 + k];
                    } else if (t + 1 < ntiles) {
                        __syncthreads();                                        // tile t + 1 is in LDS
#pragma unroll
                        for (int k = 0; k < 4; k++) nxt[k] = trow16n[k];
                    }
                    np_add_f16x32(run, cur[0], cur[1], cur[2], cur[3]);
#pragma unroll
                    for (int k = 0; k < 4; k++) cur[k] = nxt[k];
                }
            }
        }
        for (uint32_t t = 0; !H16 && t < ntiles; t++) {
            __syncthreads();                                                    // tile t is in LDS
            // fixed trip count (tiles are zero padded): LDS reads of the next 32 values are issued before the 32 dependent
            // adds of the current ones
            const float4* trow = reinterpret_cast<const float4*>(tile[t & 1][wsum][wrow]);
            float4 cur[8], nxt[8];
#pragma unroll
            for (int k = 0; k < 8; k++) cur[k] = trow[k];
#pragma unroll
            for (int c = 0; c < TC / 32; c++) {
                if (c + 1 < TC / 32) {
#pragma unroll
                    for (int k = 0; k < 8; k++) nxt[k] = trow[(c + 1) * 8 + k];
                }
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    run += cur[k].x; run += cur[k].y; run += cur[k].z; run += cur[k].w;
                }
#pragma unroll
                for (int k = 0; k < 8; k++) cur[k] = nxt[k];
            }
        }
        if (publish) sums[wsum][wrow] = run;
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();                                                        // sums published
        if (threadIdx.x < nrows) {
            const RowStats<T> st = finish_stats<T, KIND>(KIND == NORM_LAYER ? sums[NSUM - 1][threadIdx.x] : 0.0f, sums[0][threadIdx.x],
                                                         cols, eps);
            s_mu[threadIdx.x] = st.mu;
            s_r[threadIdx.x] = st.r;
        }
        __syncthreads();                                                        // row statistics published
        return;
    }

    // -------------------------------------------------------------------- waves 1..4: loads, widening, second pass
    const uint32_t lt = threadIdx.x - 64;
    const uint32_t r = lt >> 5, cv = lt & 31;                                   // row, vector within the tile
    const bool rvalid = r < nrows;
    const T* xrow = x + (row0 + (rvalid ? r : 0)) * cols;
    v4u pre0 = {0, 0, 0, 0}, pre1 = {0, 0, 0, 0};
    v4u* keep_x = np_keep;
    v4u* keep_scale = np_keep + ntiles * 256;
    v4u* keep_bias = keep_scale + ntiles * 32;

    auto issue = [&](uint32_t t, v4u& dst) {
        const uint32_t col = t * TC + cv * 8;
        if (rvalid && t < ntiles && col < cols) dst = *reinterpret_cast<const v4u*>(xrow + col);
    };
    auto step = [&](uint32_t t, v4u& reg) {
        const uint32_t buf = t & 1;
        const uint32_t col = t * TC + cv * 8;
        if (H16 && rvalid) {
            v4u sqv = {0, 0, 0, 0}, xvv = {0, 0, 0, 0};                         // past the end of the row: +0.0 terms
            if (col < cols) {
                xvv = __builtin_bit_cast(v4u, reg);
                if (KEEP) keep_x[t * 256 + lt] = xvv;                           // read back by this same thread after the walk
                const np_h8 h = __builtin_bit_cast(np_h8, xvv);
                sqv = __builtin_bit_cast(v4u, h * h);                           // T(x*x): eight f16 products, each rounded once
            }
            *reinterpret_cast<v4u*>(&tile16[buf][0][r][cv * 8]) = sqv;
            if (KIND == NORM_LAYER) *reinterpret_cast<v4u*>(&tile16[buf][NSUM - 1][r][cv * 8]) = xvv;
        } else if (rvalid) {
            float sq[8], xv[8];
            if (col < cols) {
                Vec16<T> in;
                in.u = __builtin_bit_cast(v4u, reg);
                if (KEEP) keep_x[t * 256 + lt] = in.u;                          // read back by this same thread after the walk
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    sq[q] = Ar<T>::widen(Ar<T>::mul(in.e[q], in.e[q]));
                    xv[q] = Ar<T>::widen(in.e[q]);
                }
            } else {
                // past the end of the row: +0.0 terms leave the running sums unchanged, so the walk needs no tail logic
#pragma unroll
                for (int q = 0; q < 8; q++) sq[q] = xv[q] = 0.0f;
            }
            float4* d0 = reinterpret_cast<float4*>(&tile[buf][0][r][cv * 8]);
            d0[0] = make_float4(sq[0], sq[1], sq[2], sq[3]);
            d0[1] = make_float4(sq[4], sq[5], sq[6], sq[7]);
            if (KIND == NORM_LAYER) {
                float4* d1 = reinterpret_cast<float4*>(&tile[buf][NSUM - 1][r][cv * 8]);
                d1[0] = make_float4(xv[0], xv[1], xv[2], xv[3]);
                d1[1] = make_float4(xv[4], xv[5], xv[6], xv[7]);
            }
        }
        issue(t + 2, reg);
        __syncthreads();
    };

    issue(0, pre0);
    issue(1, pre1);
    if (KEEP) {
        // scale and bias, once per block, in flight together with the first two tiles; the barriers of the walk make
        // them visible long before the output pass
        for (uint32_t c = lt; c < cols / 8; c += 256) {
            keep_scale[c] = reinterpret_cast<const v4u*>(scale)[c];
            if (KIND == NORM_LAYER && bias) keep_bias[c] = reinterpret_cast<const v4u*>(bias)[c];
        }
    }
    for (uint32_t t = 0; t < ntiles; t += 2) {
        step(t, pre0);
        if (t + 1 < ntiles) step(t + 1, pre1);
    }
    __syncthreads();                                                            // sums published (wave 0 finishes the stats)
    __syncthreads();                                                            // row statistics published
    if (!rvalid) return;
    RowStats<T> st;
    st.mu = s_mu[r];
    st.r = s_r[r];
    T* yrow = y + (row0 + r) * cols;
    const uint32_t cvec = cols / 8;
    if (KEEP) {
#pragma unroll 2
        for (uint32_t c = cv, t = 0; c < cvec; c += 32, t++) {
            Vec16<T> in, sc, bi, out;
            in.u = keep_x[t * 256 + lt];
            sc.u = keep_scale[c];
            if (KIND == NORM_LAYER && bias) bi.u = keep_bias[c];
#pragma unroll
            for (int q = 0; q < 8; q++) out.e[q] = norm_one<T, KIND>(in.e[q], st, sc.e[q], bi.e[q], bias != nullptr);
            st_stream(reinterpret_cast<v4u*>(yrow) + c, out.u);
        }
        return;
    }
    // four vectors of the row at a time, their loads issued together ([16384,4096] f16: 75.1 -> 70.4 us, RMSNorm 69.1 -> 64.0)
    constexpr int OB = 4;
    for (uint32_t c0 = cv; c0 < cvec; c0 += 32 * OB) {
        Vec16<T> in[OB], sc[OB], bi[OB];
#pragma unroll
        for (int k = 0; k < OB; k++) {
            const uint32_t c = c0 + 32 * k;
            if (c < cvec) {
                in[k].u = ld_stream(reinterpret_cast<const v4u*>(xrow) + c);
                sc[k].u = reinterpret_cast<const v4u*>(scale)[c];
                if (KIND == NORM_LAYER && bias) bi[k].u = reinterpret_cast<const v4u*>(bias)[c];
            }
        }
#pragma unroll
        for (int k = 0; k < OB; k++) {
            const uint32_t c = c0 + 32 * k;
            if (c < cvec) {
                Vec16<T> out;
#pragma unroll
                for (int q = 0; q < 8; q++) out.e[q] = norm_one<T, KIND>(in[k].e[q], st, sc[k].e[q], bi[k].e[q], bias != nullptr);
                st_stream(reinterpret_cast<v4u*>(yrow) + c, out.u);
            }
        }
    }
}

// run += the sixteen f32 values of four vectors, left to right (as one asm statement: with ordinary adds the compiler reads
// a whole tile ahead, into 256 registers)
__device__ __forceinline__ void np_add_f32x16(float& run, const v4u& a, const v4u& b, const v4u& c, const v4u& d) {
#define NP_ADD(N) "v_add_f32 %0, %0, %" #N "\n"
    asm(NP_ADD(1) NP_ADD(2) NP_ADD(3) NP_ADD(4) NP_ADD(5) NP_ADD(6) NP_ADD(7) NP_ADD(8) NP_ADD(9) NP_ADD(10) NP_ADD(11) NP_ADD(12) NP_ADD(13)
        NP_ADD(14) NP_ADD(15) NP_ADD(16)
        : "+v"(run)
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]),
          "v"(d[0]), "v"(d[1]), "v"(d[2]), "v"(d[3]));
#undef NP_ADD
}
// The same walk for rows of 8 to NF_MAX_COLS columns as a stream: persistent blocks, one to a CU, that take groups of up to
// RB rows (8, 16 or 30) in turn.  The loader waves, one for every two rows (four in blocks of 8), keep a group's rows in registers (NT vectors a thread) from the
// load to the store, and in step t of a group, while wave 0 walks tile t, they normalise and store tile t of the group
// before and load the tile PF steps ahead, across the groups: x is read once, and reads, walk and writes go on side by
// side instead of in phases that all blocks of the chip pass at the same time.
// What bounds it: with one group per block the walk (about 2.3 ns a column, whatever is left of the chip); with several,
// memory, and in bf16 the vector instructions of the output (48 us for the [16384,3072] LayerNorm whose bytes take 31.5 at
// the rate of a large copy; f16 43).  A walker occupies its SIMD's vector unit fully with 8 rows as with 30, which is why a
// block carries up to 30 rows and a CU one block: with blocks of 8 rows, two to a CU, the same LayerNorm took 54 us in f16.
// A group takes NT steps whatever its rows hold (2, 4, 8, 12, 16 and 20 exist): 1032 columns are five tiles in eight steps.
// The LayerNorm variants of 20 steps and 30 rows hold more than their 128 registers: f16 spills 15 of them (52 bytes of
// scratch a lane), bf16 5 (20 bytes); no other one does.
// Rows of any length from 8 columns and on any element boundary: no access leaves the row; the last vector of a row is
// its last eight elements, for the walk shifted so that none of them counts twice, and written with the same values as
// the one before it where they overlap.
// A row's vector is 16 bytes at `base + offset` through a buffer descriptor of the group's rows; where there is nothing to
// load or to store (columns past the end, rows past the end, the group before the first) the offset lies outside of it and
// the access is dropped, which keeps the step free of branches around memory instructions: the compiler then counts
// exactly how many may stay in flight at each wait.
constexpr uint32_t NF_MAX_COLS = 5120;                       // 20 vectors a thread
template <typename T, int KIND, int NT, int RB>
__global__ void __launch_bounds__(64 + RB * 32) norm_flow16_kernel(const T* x, const T* __restrict__ scale, const T* __restrict__ bias, T* y,
                                                               uint64_t rows, uint32_t cols, uint32_t groups, uint32_t R, float eps) {
    constexpr int TC = 256, PAD = 4, PAD16 = 8;
    constexpr int PF = 2;                                      // tiles loaded ahead; a group's step t uses slot t % PF
    constexpr int NSUM = (KIND == NORM_LAYER) ? 2 : 1;
    constexpr bool H16 = std::is_same<T, half_t>::value;                         // 16-bit tiles and the fma_mix chain
    constexpr int PITCH = H16 ? (TC + PAD16) * 2 / 16 : (TC + PAD) * 4 / 16;     // of a tile row, in 16-byte vectors
    constexpr int NW = H16 ? 4 : 8;                                              // vectors that hold 32 values
    static_assert(NT % 2 == 0 && NT % PF == 0, "the two tile buffers and the load slots are those of the same step in every group");
    __shared__ v4u tile[2][NSUM][RB][PITCH];                                     // [.][0] = squares, [.][1] = values
    __shared__ float sums[2][NSUM][RB];                                          // of the block's even and odd groups
    extern __shared__ __attribute__((aligned(16))) v4u nf_affine[];              // [ntiles * 32] scale, the same of bias
    const uint32_t ntiles = (cols + TC - 1) / TC, nvec = (cols + 7) / 8;         // ntiles <= NT; steps beyond it are empty
    const uint32_t n_mine = (groups - blockIdx.x + gridDim.x - 1) / gridDim.x;   // groups of this block: blockIdx.x, + gridDim.x, ...

    // Barriers: one per step (tile t is in LDS; wave 0 passes the one of step t + 1 when it has read all of tile t) and one
    // at the end (the last group's sums are published).
    if (threadIdx.x < 64) {
        // ---------------------------------------------------------------- wave 0: the sequential sums
        __builtin_amdgcn_s_setprio(3);
        const uint32_t wrow = threadIdx.x % RB, wsum = (threadIdx.x / RB) % NSUM;   // lanes beyond NSUM * RB shadow and never publish
        for (uint32_t it = 0; it < n_mine; it++) {
            float run = 0.0f;
            __syncthreads();                                                    // tile 0 is in LDS
            v4u cur[NW], nxt[NW];
#pragma unroll
            for (int k = 0; k < NW; k++) cur[k] = nxt[k] = tile[0][wsum][wrow][k];
            for (uint32_t t = 0; t < ntiles; t++) {
                const v4u* here = tile[t & 1][wsum][wrow];
                const v4u* next = tile[(t + 1) & 1][wsum][wrow];
#pragma unroll
                for (int c = 0; c < TC / 32; c++) {
                    if (c + 1 < TC / 32) {
#pragma unroll
                        for (int k = 0; k < NW; k++) nxt[k] = here[(c + 1) * NW + k];
                    } else if (t + 1 < ntiles) {
                        // taken before the tile's last 32 adds, whose operands are in registers: the chain does not wait
                        // for LDS at the next tile's start
                        __syncthreads();                                        // tile t + 1 is in LDS
#pragma unroll
                        for (int k = 0; k < NW; k++) nxt[k] = next[k];
                    }
                    if constexpr (H16) {
                        np_add_f16x32(run, cur[0], cur[1], cur[2], cur[3]);
                    } else {
#pragma unroll
                        for (int k = 0; k < NW; k += 4) np_add_f32x16(run, cur[k], cur[k + 1], cur[k + 2], cur[k + 3]);
                    }
#pragma unroll
                    for (int k = 0; k < NW; k++) cur[k] = nxt[k];
                }
            }
            if (threadIdx.x < NSUM * RB) sums[it & 1][wsum][wrow] = run;
            for (uint32_t t = ntiles; t < (uint32_t)NT; t++) __syncthreads();   // the empty steps
        }
        __syncthreads();                                                        // the last group's sums are published
        return;
    }

    // -------------------------------------------------------------------- the other waves: load, square, normalise, store
    const uint32_t lt = threadIdx.x - 64;
    const uint32_t r = lt >> 5, cv = lt & 31;                                   // row, vector within the tile
    const uint32_t row_bytes = cols * 2;
    constexpr uint32_t OOB = 0x80000000u;
    const uint32_t last = ntiles - 1;
    // This thread's vector of a tile: where it starts in its row, in bytes from the tile's first column.  In a row's last
    // tile the last vector starts eight elements before the row's end, and there is none behind it.
    const uint32_t tail_col = last * TC + cv * 8;
    const uint32_t off_main = cv * 16;
    const uint32_t off_tail = tail_col >= cols ? OOB : ((tail_col + 8 > cols ? cols - 8 : tail_col) - last * TC) * 2;
    const uint32_t drop = tail_col < cols && tail_col + 8 > cols ? tail_col + 8 - cols : 0u;    // its elements that the vector before holds too
    // of tile t: its first column is added last (it may take an `off_tail` from before the tile back into the row)
    auto pick = [&](uint32_t t, uint32_t row, uint32_t row_tail) -> uint32_t {
        uint32_t l = last;
        asm volatile("" : "+s"(l));                                             // compared afresh: kept in registers, the masks of all steps would spill
        return (t < l ? row : t == l ? row_tail : OOB) + t * (TC * 2);
    };
    struct Group {                                                              // the same for the whole block but for `row`
        const T* x;                                                             // 16-byte boundary at or before the first row
        T* y;
        uint32_t bytes_x, bytes_y;                                              // from there to the last row's end
        uint32_t row_x, row_y, tail_x, tail_y;                                  // this thread's vector in tile 0 and in the last one (less its columns), or OOB
    };
    auto group_of = [&](uint32_t it) -> Group {
        Group g;
        const uint64_t row0 = ((uint64_t)blockIdx.x + (uint64_t)it * gridDim.x) * R;
        const bool ok = it < n_mine;
        const uint32_t nrows = !ok ? 0u : rows - row0 < (uint64_t)R ? (uint32_t)(rows - row0) : R;
        const T* gx = x + (ok ? row0 : 0) * cols;
        T* gy = y + (ok ? row0 : 0) * cols;
        const uint32_t sx = (uint32_t)((uintptr_t)gx & 15u), sy = (uint32_t)((uintptr_t)gy & 15u);
        g.x = reinterpret_cast<const T*>(reinterpret_cast<const char*>(gx) - sx);
        g.y = reinterpret_cast<T*>(reinterpret_cast<char*>(gy) - sy);
        g.bytes_x = sx + nrows * row_bytes;
        g.bytes_y = sy + nrows * row_bytes;
        const bool have = r < nrows, have_tail = have && off_tail != OOB;
        g.row_x = have ? sx + r * row_bytes + off_main : OOB;
        g.row_y = have ? sy + r * row_bytes + off_main : OOB;
        g.tail_x = have_tail ? sx + r * row_bytes + off_tail : OOB;
        g.tail_y = have_tail ? sy + r * row_bytes + off_tail : OOB;
        return g;
    };
    auto load = [&](const Group& g, uint32_t t) -> v4u {
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(g.x), 0, g.bytes_x, 0x00020000);
        return __builtin_amdgcn_raw_buffer_load_b128(rx, pick(t, g.row_x, g.tail_x), 0, 2);            // 2: non-temporal
    };
    Group cur = group_of(0), nxt = group_of(1), prev = group_of(n_mine);        // prev: no rows, its stores are dropped
    v4u pre[PF], held[NT];
#pragma unroll
    for (int k = 0; k < PF; k++) pre[k] = load(cur, k);
    for (uint32_t c = lt; c < nvec; c += blockDim.x - 64) {
        const uint32_t at = c * 8 + 8 > cols ? cols - 8 : c * 8;
        v4u v;
        __builtin_memcpy(&v, scale + at, 16);
        nf_affine[c] = v;
        if (KIND == NORM_LAYER) {                                               // without a bias -0, which changes no value that it is added to
            v = v4u{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
            if (bias) __builtin_memcpy(&v, bias + at, 16);
            nf_affine[ntiles * (TC / 8) + c] = v;
        }
    }
#pragma unroll
    for (int t = 0; t < NT; t++) held[t] = v4u{0u, 0u, 0u, 0u};
    RowStats<T> st;
    st.mu = st.r = Ar<T>::conv(0.0f);
    auto put = [&](int t) {                                                     // tile t of the group before
        const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(prev.y, 0, prev.bytes_y, 0x00020000);
        uint32_t l = last, c = cv;                                              // opaque: else all of scale and bias is kept in registers across the groups
        asm volatile("" : "+s"(l), "+v"(c));
        c += ((uint32_t)t < l ? (uint32_t)t : l) * (TC / 8);
        const v4u sc = nf_affine[c], bi = KIND == NORM_LAYER ? nf_affine[ntiles * (TC / 8) + c] : v4u{0u, 0u, 0u, 0u};
        const v4u out = norm_vec16<T, KIND>(held[t], st, sc, bi);
        __builtin_amdgcn_raw_buffer_store_b128(out, ry, pick(t, prev.row_y, prev.tail_y), 0, 2);
    };
    for (uint32_t it = 0; it < n_mine; it++) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const v4u mine = pre[t % PF];                                       // zeros past the row's end: +0.0 terms leave the running sums
            uint32_t l = last;
            asm volatile("" : "+s"(l));
            if ((uint32_t)t <= l) {
                v4u xv = mine;
                if ((uint32_t)t == l) {                                         // only the elements that the vector before does not hold
                    if (drop & 1) xv = v4u{(xv[0] >> 16) | (xv[1] << 16), (xv[1] >> 16) | (xv[2] << 16), (xv[2] >> 16) | (xv[3] << 16), xv[3] >> 16};
                    if (drop & 2) xv = v4u{xv[1], xv[2], xv[3], 0u};
                    if (drop & 4) xv = v4u{xv[2], xv[3], 0u, 0u};
                }
                if constexpr (H16) {
                    const np_h8 h = __builtin_bit_cast(np_h8, xv);
                    tile[t & 1][0][r][cv] = __builtin_bit_cast(v4u, h * h);     // T(x*x): eight f16 products, each rounded once
                    if (KIND == NORM_LAYER) tile[t & 1][NSUM - 1][r][cv] = xv;
                } else {
                    v4u sq[2], wide[2];
#pragma unroll
                    for (int w = 0; w < 4; w++) {
                        const float lo = u2f(xv[w] << 16), hi = u2f(xv[w] & 0xffff0000u);
                        wide[w / 2][w % 2 * 2] = f2u(lo);
                        wide[w / 2][w % 2 * 2 + 1] = f2u(hi);
                        sq[w / 2][w % 2 * 2] = f2u(np_round_bf16(lo * lo));
                        sq[w / 2][w % 2 * 2 + 1] = f2u(np_round_bf16(hi * hi));
                    }
                    tile[t & 1][0][r][cv * 2] = sq[0];
                    tile[t & 1][0][r][cv * 2 + 1] = sq[1];
                    if (KIND == NORM_LAYER) {
                        tile[t & 1][NSUM - 1][r][cv * 2] = wide[0];
                        tile[t & 1][NSUM - 1][r][cv * 2 + 1] = wide[1];
                    }
                }
            }
            pre[t % PF] = t + PF < NT ? load(cur, t + PF) : load(nxt, t + PF - NT);
            __syncthreads();                                                    // tile t is in LDS; with t = 0 the sums of the group before
            if (t == 0)
                st = finish_stats<T, KIND>(KIND == NORM_LAYER ? sums[(it & 1) ^ 1][NSUM - 1][r] : 0.0f, sums[(it & 1) ^ 1][0][r], cols, eps);
            put(t);
#pragma unroll
            for (int w = 0; w < 4; w++) asm volatile("v_mov_b32 %0, %1" : "+v"(held[t][w]) : "v"(mine[w]));
            __builtin_amdgcn_sched_barrier(0);
        }
        prev = cur;
        cur = nxt;
        nxt = group_of(it + 2);
    }
    __syncthreads();                                                            // the last group's sums are published
    st = finish_stats<T, KIND>(KIND == NORM_LAYER ? sums[(n_mine & 1) ^ 1][NSUM - 1][r] : 0.0f, sums[(n_mine & 1) ^ 1][0][r], cols, eps);
#pragma unroll
    for (int t = 0; t < NT; t++) {
        put(t);
        if (t % 3 == 2) __builtin_amdgcn_sched_barrier(0);                      // not all of scale and bias at once
    }
}

// ------------------------------------------------------------------------------------------------------------------
// GroupNorm in slices (gn_reg_kernel below takes what fits a block).  x is [B, C, L] contiguous, so group (b, g) is one contiguous run of
// glen = (C/G)*L elements.
// stats kernel: grid (B*G, splits); block s of a group reduces elements [s*chunk, min((s+1)*chunk, glen)) to
//               (mean, M2, count) with a two-pass local variance (second pass re-reads the slice from cache).
// apply kernel: same grid; every block combines the group's partials (Chan et al.), then normalises its slice:
//               y = (x - mean) * rstd * w[c] + b[c], f32 arithmetic, rounded to T once.
// ------------------------------------------------------------------------------------------------------------------
// The f32 arithmetic of GroupNorm on an element as it was loaded: the widening of an f16 operand is part of the fused
// multiply-add (v_fma_mix_f32), so an f16 element costs one instruction for the mean, two for the variance and three for the output
// where widening, adding, multiplying and rounding one by one cost 2, 4 and 6.  1 * e + acc rounds as e + acc does; the squares and
// the last multiplication are rounded once less than as separate operations.
template <typename T> __device__ __forceinline__ float gn_plus(T e, float acc) {
    if constexpr (std::is_same<T, half_t>::value) return __builtin_fmaf((float)e, 1.0f, acc);
    else return Ar<T>::widen(e) + acc;
}
template <typename T> __device__ __forceinline__ float gn_dev2(T e, float mean, float acc) {
    const float d = gn_plus<T>(e, -mean);
    return __builtin_fmaf(d, d, acc);
}

// VE = elements per access: 16 / sizeof(T) on the vector path (slices, groups and base pointers are multiples of it), 1 otherwise
template <typename T, int VE>
__global__ void __launch_bounds__(BLOCK) gn_stats_kernel(const T* __restrict__ x, float* __restrict__ part, uint32_t glen,
                                                         uint32_t chunk, uint32_t splits) {
    __shared__ float red[WAVES];
    __shared__ float bc;
    const uint32_t s = blockIdx.y, grp = blockIdx.x;
    const T* xs = x + (uint64_t)grp * glen;
    const uint32_t c0 = s * chunk;
    const uint32_t c1 = (c0 + chunk < glen) ? c0 + chunk : glen;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    float acc = 0.0f;
    for (uint32_t i = c0 + threadIdx.x * VE; i < c1; i += BLOCK * VE) {
        if (VE > 1) {
            Vec16<T> v;
            v.u = *reinterpret_cast<const v4u*>(xs + i);
#pragma unroll
            for (int q = 0; q < VE; q++) acc = gn_plus<T>(v.e[q], acc);
        } else {
            acc = gn_plus<T>(xs[i], acc);
        }
    }
    acc = wave_sum(acc);
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.0f;
        for (int w = 0; w < WAVES; w++) t += red[w];
        bc = t / (float)(c1 - c0);
    }
    __syncthreads();
    const float mean = bc;
    float m2 = 0.0f;
    for (uint32_t i = c0 + threadIdx.x * VE; i < c1; i += BLOCK * VE) {     // second pass: the slice is in cache
        if (VE > 1) {
            Vec16<T> v;
            v.u = *reinterpret_cast<const v4u*>(xs + i);
#pragma unroll
            for (int q = 0; q < VE; q++) m2 = gn_dev2<T>(v.e[q], mean, m2);
        } else {
            m2 = gn_dev2<T>(xs[i], mean, m2);
        }
    }
    m2 = wave_sum(m2);
    __syncthreads();
    if (lane == 0) red[wave] = m2;
    __syncthreads();
    if (threadIdx.x == 0) {
        float t = 0.0f;
        for (int w = 0; w < WAVES; w++) t += red[w];
        float* o = part + ((uint64_t)grp * splits + s) * 3;
        o[0] = mean;
        o[1] = t;
        o[2] = (float)(c1 - c0);
    }
}

// The same partials from a slice that the block's registers hold (NV vectors a thread): the slice is read once, with all
// its loads in flight together, and the second pass runs on registers ([16,256,4096] f32, slices of 32 KiB: 49.7 -> 33.8 us for the two launches).
template <typename T, int NV>
__global__ void __launch_bounds__(BLOCK) gn_stats_reg_kernel(const T* __restrict__ x, float* __restrict__ part, uint32_t glen,
                                                             uint32_t chunk, uint32_t splits) {
    constexpr int VE = 16 / sizeof(T);
    __shared__ float red[WAVES];
    const uint32_t s = blockIdx.y, grp = blockIdx.x;
    const uint32_t c0 = s * chunk;
    const uint32_t c1 = (c0 + chunk < glen) ? c0 + chunk : glen;
    const v4u* xs = reinterpret_cast<const v4u*>(x + (uint64_t)grp * glen + c0);
    const uint32_t nvec = (c1 - c0) / VE;
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    Vec16<T> v[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = threadIdx.x + k * BLOCK;
        v[k].u = v4u{0u, 0u, 0u, 0u};
        if (i < nvec) v[k].u = xs[i];
    }
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; k++) {
#pragma unroll
        for (int q = 0; q < VE; q++) acc = gn_plus<T>(v[k].e[q], acc);             // vectors past the slice hold zeros
    }
    acc = wave_sum(acc);
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; w++) t += red[w];
    const float mean = t / (float)(c1 - c0);
    float m2 = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        if (threadIdx.x + k * BLOCK < nvec) {
#pragma unroll
            for (int q = 0; q < VE; q++) m2 = gn_dev2<T>(v[k].e[q], mean, m2);
        }
    }
    m2 = wave_sum(m2);
    __syncthreads();
    if (lane == 0) red[wave] = m2;
    __syncthreads();
    if (threadIdx.x == 0) {
        float u = 0.0f;
        for (int w = 0; w < WAVES; w++) u += red[w];
        float* o = part + ((uint64_t)grp * splits + s) * 3;
        o[0] = mean;
        o[1] = u;
        o[2] = (float)(c1 - c0);
    }
}

// y = (x - mean) * rstd * w[c] + b[c] for the VE elements of one vector that starts at element e0 of its group, whose first
// channel is cbase.  With L a multiple of VE the vector lies in one channel; a vector of longer rows lies in at most two (both
// are read ahead and chosen element by element), and where L < VE the channel is stepped.
template <typename T>
__device__ __forceinline__ v4u gn_affine_vec(const Vec16<T>& v, uint32_t e0, uint32_t cbase, FastDiv L, const T* __restrict__ scale,
                                             const T* __restrict__ bias, float mean, float rstd) {
    constexpr int VE = 16 / sizeof(T);
    Vec16<T> o;
    const uint32_t ch = fd_div(e0, L);
    uint32_t c = cbase + ch;
    if (L.d % VE == 0) {
        const float w = scale ? Ar<T>::widen(scale[c]) : 1.0f;
        const float b = bias ? Ar<T>::widen(bias[c]) : 0.0f;
#pragma unroll
        for (int q = 0; q < VE; q++) o.e[q] = Ar<T>::conv(__builtin_fmaf(gn_plus<T>(v.e[q], -mean) * rstd, w, b));
    } else if (L.d >= VE) {
        const uint32_t left = L.d - (e0 - ch * L.d);                       // elements of the vector in channel c, if fewer than VE
        const uint32_t c1 = left < (uint32_t)VE ? c + 1 : c;
        const float w0 = scale ? Ar<T>::widen(scale[c]) : 1.0f, w1 = scale ? Ar<T>::widen(scale[c1]) : 1.0f;
        const float b0 = bias ? Ar<T>::widen(bias[c]) : 0.0f, b1 = bias ? Ar<T>::widen(bias[c1]) : 0.0f;
#pragma unroll
        for (int q = 0; q < VE; q++)
            o.e[q] = Ar<T>::conv(__builtin_fmaf(gn_plus<T>(v.e[q], -mean) * rstd, (uint32_t)q < left ? w0 : w1, (uint32_t)q < left ? b0 : b1));
    } else {
        uint32_t r = e0 - ch * L.d;
#pragma unroll
        for (int q = 0; q < VE; q++) {
            const float w = scale ? Ar<T>::widen(scale[c]) : 1.0f;
            const float b = bias ? Ar<T>::widen(bias[c]) : 0.0f;
            o.e[q] = Ar<T>::conv(__builtin_fmaf(gn_plus<T>(v.e[q], -mean) * rstd, w, b));
            if (++r == L.d) {
                r = 0;
                c++;
            }
        }
    }
    return o.u;
}

// Combines the partials of one group (Chan et al.) in double, by the first wave of the block: lane k takes partial k (the
// launcher keeps splits <= 64 here), then a tree over the wave, in the same order in every block of the group.
__device__ __forceinline__ void gn_combine_wave(const float* __restrict__ p, uint32_t splits, float eps, float& s_mean, float& s_rstd) {
    if (threadIdx.x >= WAVE) return;
    double n = 0.0, mean = 0.0, m2 = 0.0;
    if (threadIdx.x < splits) {
        mean = (double)p[3 * threadIdx.x];
        m2 = (double)p[3 * threadIdx.x + 1];
        n = (double)p[3 * threadIdx.x + 2];
    }
    for (int off = WAVE / 2; off > 0; off >>= 1) {
        const double nb = __shfl_down(n, off), mb = __shfl_down(mean, off), m2b = __shfl_down(m2, off);
        if (nb != 0.0) {
            const double nt = n + nb;
            const double delta = mb - mean;
            mean += delta * (nb / nt);
            m2 += m2b + delta * delta * (n * nb / nt);
            n = nt;
        }
    }
    if (threadIdx.x == 0) {
        s_mean = (float)mean;
        s_rstd = (float)(1.0 / sqrt(m2 / n + (double)eps));
    }
}

template <typename T, int VE>
__global__ void __launch_bounds__(BLOCK) gn_apply_kernel(const T* __restrict__ x, const T* __restrict__ scale,
                                                         const T* __restrict__ bias, T* __restrict__ y,
                                                         const float* __restrict__ part, uint32_t glen, uint32_t chunk, uint32_t splits,
                                                         uint32_t cpg, uint32_t groups, FastDiv L, float eps) {
    __shared__ float s_mean, s_rstd;
    const uint32_t s = blockIdx.y, grp = blockIdx.x;
    gn_combine_wave(part + (uint64_t)grp * splits * 3, splits, eps, s_mean, s_rstd);
    __syncthreads();
    const float meanf = s_mean, rstd = s_rstd;
    const uint32_t g = grp % groups;
    const T* xs = x + (uint64_t)grp * glen;
    T* ys = y + (uint64_t)grp * glen;
    const uint32_t c0 = s * chunk;
    const uint32_t c1 = (c0 + chunk < glen) ? c0 + chunk : glen;
    for (uint32_t i = c0 + threadIdx.x * VE; i < c1; i += BLOCK * VE) {
        if (VE > 1) {
            Vec16<T> v;
            v.u = *reinterpret_cast<const v4u*>(xs + i);
            st_stream(reinterpret_cast<v4u*>(ys + i), gn_affine_vec<T>(v, i, g * cpg, L, scale, bias, meanf, rstd));
        } else {
            const uint32_t c = g * cpg + fd_div(i, L);
            const float w = scale ? Ar<T>::widen(scale[c]) : 1.0f;
            const float b = bias ? Ar<T>::widen(bias[c]) : 0.0f;
            ys[i] = Ar<T>::conv(__builtin_fmaf(gn_plus<T>(xs[i], -meanf) * rstd, w, b));
        }
    }
}

// gn_apply_kernel for slices of up to NV vectors a thread: all loads of the slice are in flight before the first is used
template <typename T, int NV>
__global__ void __launch_bounds__(BLOCK) gn_apply_reg_kernel(const T* __restrict__ x, const T* __restrict__ scale,
                                                             const T* __restrict__ bias, T* __restrict__ y,
                                                             const float* __restrict__ part, uint32_t glen, uint32_t chunk,
                                                             uint32_t splits, uint32_t cpg, uint32_t groups, FastDiv L, float eps) {
    constexpr int VE = 16 / sizeof(T);
    __shared__ float s_mean, s_rstd;
    const uint32_t s = blockIdx.y, grp = blockIdx.x;
    const uint32_t c0 = s * chunk;
    const uint32_t c1 = (c0 + chunk < glen) ? c0 + chunk : glen;
    const v4u* xs = reinterpret_cast<const v4u*>(x + (uint64_t)grp * glen + c0);
    v4u* ys = reinterpret_cast<v4u*>(y + (uint64_t)grp * glen + c0);
    const uint32_t nvec = (c1 - c0) / VE;
    Vec16<T> v[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = threadIdx.x + k * BLOCK;
        v[k].u = v4u{0u, 0u, 0u, 0u};
        if (i < nvec) v[k].u = ld_stream(xs + i);
    }
    gn_combine_wave(part + (uint64_t)grp * splits * 3, splits, eps, s_mean, s_rstd);
    __syncthreads();
    const float meanf = s_mean, rstd = s_rstd;
    const uint32_t g = grp % groups;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = threadIdx.x + k * BLOCK;
        if (i < nvec) {
            st_stream(ys + i, gn_affine_vec<T>(v[k], c0 + i * VE, g * cpg, L, scale, bias, meanf, rstd));
        }
    }
}

template <typename T, int KIND, bool SPAN>
int launch_norm_wave(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols, float eps);

template <typename T, int KIND>
int launch_norm(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols, float eps) {
    constexpr int VE = 16 / sizeof(T);
    const bool io_aligned = rt_aligned(x, 16) && rt_aligned(y, 16);
    constexpr uint32_t MAX_VEC = NORM_WIDE_BLOCK * 16;       // 65536 f32 columns
    if (io_aligned && cols % VE == 0 && rt_aligned(scale, 16) && (!bias || rt_aligned(bias, 16)) && cols / VE <= MAX_VEC)
        return launch_norm_wave<T, KIND, false>(dev, x, scale, bias, y, rows, cols, eps);
    // rows that are not whole vectors (or scale / bias off their alignment): over the aligned vectors that cover each row
    if (io_aligned && (cols + 2 * VE - 2) / VE <= MAX_VEC)
        return launch_norm_wave<T, KIND, true>(dev, x, scale, bias, y, rows, cols, eps);
    RT_REQUIRE(rows <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
    hipLaunchKernelGGL((norm_generic_kernel<T, KIND>), dim3((unsigned)rows), dim3(BLOCK), 0, dev->stream, (const T*)x, (const T*)scale,
                       (const T*)bias, (T*)y, rows, cols, eps);
    RT_CHECK_LAUNCH("norm_generic_kernel");
    return RT_OK;
}

template <typename T, int KIND, bool SPAN>
int launch_norm_wave(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols, float eps) {
    constexpr int VE = 16 / sizeof(T);
    const uint32_t nvec = SPAN ? (cols + 2 * VE - 2) / VE : cols / VE;       // SPAN: the most vectors a row can touch
    if (nvec <= 32) {
        // rows of at most 32 vectors: a group of 2..32 lanes per row (one vector each), so that a wave carries 2..32 rows
        // and as many bytes as with long rows
        const uint32_t lanes = nvec <= 2 ? 2 : nvec <= 4 ? 4 : nvec <= 8 ? 8 : nvec <= 16 ? 16 : 32;
        const uint64_t blocks = (rows + BLOCK / lanes - 1) / (BLOCK / lanes);
        RT_REQUIRE(blocks <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
        const dim3 grid((unsigned)blocks), block(BLOCK);
#define RT_NARROW(L) hipLaunchKernelGGL((norm_wave_kernel<T, 1, KIND, L, SPAN>), grid, block, 0, dev->stream, (const T*)x, (const T*)scale, (const T*)bias, (T*)y, rows, cols, eps)
        if (lanes == 2) RT_NARROW(2);
        else if (lanes == 4) RT_NARROW(4);
        else if (lanes == 8) RT_NARROW(8);
        else if (lanes == 16) RT_NARROW(16);
        else RT_NARROW(32);
#undef RT_NARROW
        RT_CHECK_LAUNCH("norm_wave_kernel");
        return RT_OK;
    }
    if (nvec <= (uint32_t)(WAVE * 8)) {
        const uint32_t nv = (nvec + WAVE - 1) / WAVE;
        const uint64_t blocks = (rows + WAVES - 1) / WAVES;
        RT_REQUIRE(blocks <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
        const dim3 grid((unsigned)blocks), block(BLOCK);
#define RT_NORM(NVC)                                                                                                                 \
    hipLaunchKernelGGL((norm_wave_kernel<T, NVC, KIND, WAVE, SPAN>), grid, block, 0, dev->stream, (const T*)x, (const T*)scale, (const T*)bias, \
                       (T*)y, rows, cols, eps)
        if (nv <= 1) RT_NORM(1);
        else if (nv <= 2) RT_NORM(2);
        else if (nv <= 3) RT_NORM(3);
        else if (nv <= 4) RT_NORM(4);
        else if (nv <= 5) RT_NORM(5);
        else if (nv <= 6) RT_NORM(6);
        else RT_NORM(8);
#undef RT_NORM
        RT_CHECK_LAUNCH("norm_wave_kernel");
        return RT_OK;
    }
    RT_REQUIRE(rows <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
    if (nvec <= (uint32_t)(BLOCK * 8)) {                     // longer rows: the 256 threads of a block share one row
        const uint32_t nv = (nvec + BLOCK - 1) / BLOCK;
        const dim3 grid((unsigned)rows), block(BLOCK);
#define RT_NORM(NVC)                                                                                                                  \
    hipLaunchKernelGGL((norm_wave_kernel<T, NVC, KIND, BLOCK, SPAN>), grid, block, 0, dev->stream, (const T*)x, (const T*)scale, (const T*)bias, \
                       (T*)y, rows, cols, eps)
        if (nv <= 3) RT_NORM(3);
        else if (nv <= 4) RT_NORM(4);
        else if (nv <= 6) RT_NORM(6);
        else RT_NORM(8);
#undef RT_NORM
    } else {                                                 // up to 65536 f32 columns (the caller has checked): 1024 threads share one row
        const uint32_t nv = (nvec + NORM_WIDE_BLOCK - 1) / NORM_WIDE_BLOCK;
        const dim3 grid((unsigned)rows), block(NORM_WIDE_BLOCK);
#define RT_NORM(NVC)                                                                                                                  \
    hipLaunchKernelGGL((norm_wave_kernel<T, NVC, KIND, NORM_WIDE_BLOCK, SPAN>), grid, block, 0, dev->stream, (const T*)x, (const T*)scale, \
                       (const T*)bias, (T*)y, rows, cols, eps)
        if (nv <= 4) RT_NORM(4);
        else if (nv <= 8) RT_NORM(8);
        else if (nv <= 13) RT_NORM(13);
        else RT_NORM(16);
#undef RT_NORM
    }
    RT_CHECK_LAUNCH("norm_wave_kernel");
    return RT_OK;
}

// 16-bit reference arithmetic, many rows of at most 128 columns (whole aligned vectors): one lane per row.  A block's
// 256 rows are one contiguous run that passes through LDS with coalesced 16-byte accesses (row pitch 16 bytes more than
// the row, so neighbouring lanes' LDS accesses fall into different banks); the sequential f32 sums are short chains
// inside the lane.  (The tile walker above carries 8 rows per block however short they are: a million rows of 8 columns
// took it 479 us.)
template <typename T, int KIND, int NV>
__global__ void __launch_bounds__(BLOCK) norm16_lane_kernel(const T* x, const T* __restrict__ scale, const T* __restrict__ bias, T* y,
                                                            uint64_t rows, float eps) {
    __shared__ v4u stage[BLOCK * (NV + 1)];
    const uint64_t row0 = (uint64_t)blockIdx.x * BLOCK;
    const uint32_t nrows = rows - row0 < (uint64_t)BLOCK ? (uint32_t)(rows - row0) : (uint32_t)BLOCK;
    const v4u* xb = reinterpret_cast<const v4u*>(x) + row0 * NV;
    v4u* yb = reinterpret_cast<v4u*>(y) + row0 * NV;
    const uint32_t nvec = nrows * NV;
    for (uint32_t i = threadIdx.x; i < nvec; i += BLOCK) stage[(i / NV) * (NV + 1) + i % NV] = ld_stream(xb + i);
    __syncthreads();
    if (threadIdx.x < nrows) {
        v4u* mine = stage + threadIdx.x * (NV + 1);
        Vec16<T> v[NV];
#pragma unroll
        for (int k = 0; k < NV; k++) v[k].u = mine[k];
        float sx = 0.0f, sq = 0.0f;                          // the reference's order: element 0 first
#pragma unroll
        for (int k = 0; k < NV; k++)
#pragma unroll
            for (int q = 0; q < 8; q++) {
                sq += Ar<T>::widen(Ar<T>::mul(v[k].e[q], v[k].e[q]));
                if (KIND == NORM_LAYER) sx += Ar<T>::widen(v[k].e[q]);
            }
        const RowStats<T> st = finish_stats<T, KIND>(sx, sq, NV * 8, eps);
#pragma unroll
        for (int k = 0; k < NV; k++) {
            Vec16<T> sc, bi;
            sc.u = reinterpret_cast<const v4u*>(scale)[k];
            if (KIND == NORM_LAYER && bias) bi.u = reinterpret_cast<const v4u*>(bias)[k];
#pragma unroll
            for (int q = 0; q < 8; q++) v[k].e[q] = norm_one<T, KIND>(v[k].e[q], st, sc.e[q], bi.e[q], bias != nullptr);
            mine[k] = v[k].u;
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < nvec; i += BLOCK) st_stream(yb + i, stage[(i / NV) * (NV + 1) + i % NV]);
}

template <typename T, int KIND>
int launch_norm16_lane(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols, float eps) {
    const uint64_t blocks = (rows + BLOCK - 1) / BLOCK;
    RT_REQUIRE(blocks <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
#define RT_LANE(NV)                                                                                                              \
    case NV:                                                                                                                     \
        hipLaunchKernelGGL((norm16_lane_kernel<T, KIND, NV>), dim3((unsigned)blocks), dim3(BLOCK), 0, dev->stream, (const T*)x, \
                           (const T*)scale, (const T*)bias, (T*)y, rows, eps);                                                   \
        break
    switch (cols / 8) {
        RT_LANE(1); RT_LANE(2); RT_LANE(3); RT_LANE(4); RT_LANE(5); RT_LANE(6); RT_LANE(7); RT_LANE(8);
        RT_LANE(9); RT_LANE(10); RT_LANE(11); RT_LANE(12); RT_LANE(13); RT_LANE(14); RT_LANE(15); RT_LANE(16);
        default: return rt_fail(RT_ERR_ARG, "norm: internal: %u columns in the one-lane-per-row kernel", cols);
    }
#undef RT_LANE
    RT_CHECK_LAUNCH("norm16_lane_kernel");
    return RT_OK;
}

template <typename T, int KIND, int RB>
int launch_norm16_rb(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols, float eps) {
    const uint64_t blocks = (rows + RB - 1) / RB;
    RT_REQUIRE(blocks <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
    hipLaunchKernelGGL((norm_seq16_kernel<T, RB, KIND>), dim3((unsigned)blocks), dim3(BLOCK), 0, dev->stream, (const T*)x,
                       (const T*)scale, (const T*)bias, (T*)y, rows, cols, eps);
    RT_CHECK_LAUNCH("norm_seq16_kernel");
    return RT_OK;
}

// the steps that norm_flow16_kernel takes per group for rows of `nt` tiles
inline uint32_t nf_steps(uint32_t nt) { return nt <= 2 ? 2 : nt <= 4 ? 4 : nt <= 8 ? 8 : nt <= 12 ? 12 : nt <= 16 ? 16 : 20; }

// Where norm_flow16_kernel takes a launch.  Both sides were timed on 1 to 1 million rows, inputs and outputs moving through
// 580 MB; the figures are us, the other kernel / this one.
// Rows that are not whole aligned vectors: against norm_seq16_kernel, which reads element by element but starts a row with
// little to do.  This kernel walks whole 256-column tiles, two at least, so rows of up to 128 columns gain only in large
// numbers, and those of more than 64 also where the launch is a single round of walks (LayerNorm f16: [256,257] 9.0 / 5.5,
// [10240,257] 14.7 / 8.5, [10240,31] 5.6 / 7.5, [50000,31] 30 / 16; bf16 [10240,13] 5.9 / 10.1, RMSNorm bf16 [65536,13] 15.7 / 21.9).
inline bool nf_takes_ragged(bool bf16, bool layer, uint64_t rows, uint32_t cols, uint64_t cus) {
    if (rows < 16 && cols <= 160) return false;
    if (cols > 128) return true;
    if (cols > 64) return rows <= 16 * cus || rows >= (!bf16 ? 60 : layer ? 100 : 64) * cus || (!bf16 && !layer && cols > 96);
    if (layer) return rows >= (bf16 ? 129 : 120) * cus;
    if (!bf16) return rows >= (cols > 40 ? 60 : 120) * cus && cols >= 12;
    return (cols >= 40 && rows >= 120 * cus) || (cols >= 24 && rows > 256 * cus);
}
// Rows of whole aligned vectors: where a wave per row (rt_norm_row.hip) takes them, timed like the above but on 4 kinds of rows; us, the best of the
// others / that one, for rows of N(0, 1), and where it matters for rows with their mean taken off (c) and the same with four columns 40 times as large (o).
// It adds in any order where the ordered sum's rounding is sure without the order.  For the squares that hangs little on the rows.
//   RMSNorm bf16, nearly always sure: from 264 columns up ([256,5120] 22.0 / 10.8, [2048,2560] 9.5 / 8.6, [16384,3072] 40.7 / 37.2, [65536,384] 31.8 / 22.3).
//   RMSNorm f16, one row in ten open, 1 to 4 us a wave: up to 16 rows a CU (against a kernel that is gone: [4096,264] 7.8 / 5.7, [4096,1280] 9.1 / 7.9, [1024,5120] 18.6 / 11.3; of 3072 to
//     4096 columns and 32 to 128 rows no gain, 6.9 / 6.9, and rows whose squares are subnormal 6.6 / 7.2); then where the walk takes its rows in many
//     rounds ([16384,320] 9.6 / 8.0, [16384,1280] 21.3 / 18.0, [16384,2560] 34.3 / 32.1; [14000,1792] 19.9 / 20.9, [14000,1024] 11.8 / 13.0, [14000,640] o 10.4 / 11.3;
//     [16384,264] 9.5 / 10.1), from 3072 columns where its steps are not full ([10240,3840] 35.5 / 32.8, [16384,4608] 58.5 / 57.1; [12288,3072] 28.9 / 30.1,
//     [7200,4096] 24.3 / 26.5) or are many ([8192,5120] 37.1 / 35.5, [32768,5120] 123 / 119; [7200,5120] 29.9 / 32.1), and where it shares
//     lines between rows ([12288,4088] 46.4 / 40.7, [12288,5112] 61.6 / 50.3).
// The sum of x is small against its terms, and of rows with no mean it is nearly all rounding: f16 rows of that kind are added in order all of them, bf16 ones one
// in six, 3 us a wave for 2560 columns.  A line holds for rows of N(0, 1), c and o alike.  (Rows of values and their negatives, whose sum is zero but for the
// roundings on the way, are added in order all of them; they lose where the others gain little: bf16 [1536,1280] 9.5 / 10.8, [16384,2560] 47.6 / 59.5.)
//   LayerNorm f16: up to a row a CU, where the walk's latency is the launch and ordered rows take as long ([256,2560] 11.8 / 8.7, c 11.9 / 11.1; [16,4608] 18.5 / 10.7, c 18.5 / 17.0;
//     [256,4096] 15.6 / 15.4, c 15.6 / 16.3; [256,640] 5.4 / 4.7, c 5.4 / 5.9; [512,1280] 7.2 / 6.0, c 7.2 / 7.8), and up to 4 of one step and less
//     ([1024,384] 4.7 / 3.8, c 4.7 / 4.4; [1024,512] 4.4 / 4.2, c 4.4 / 4.9).
//   LayerNorm bf16: up to 4 rows a CU ([1024,2560] 14.6 / 8.8, c 14.5 / 11.2; [1024,5120] 22.6 / 15.5, c 22.6 / 20.5), up to 11 of up to 3072 columns
//     ([2048,2560] 14.8 / 11.6, c 14.9 / 11.9, o 14.8 / 13.7; [2816,1408] 12.2 / 9.9, c 12.3 / 10.2; but [3584,1408] c 12.6 / 12.3, o 12.5 / 13.7, [2048,4096] c 19.4 / 22.3); where three of
//     the walk's blocks fit a CU, at 16 to 24 rows ([4608,904] 15.6 / 10.4, c 15.6 / 11.7); and in large numbers where a quarter of the walk's steps is
//     empty ([9000,1408] 25.3 / 19.1, c 25.5 / 21.2, o 25.2 / 21.3; [8192,1280] 20.3 / 18.9, c 20.3 / 20.7, o 20.3 / 23.4; [8192,2560] 31.1 / 22.4, c 30.8 / 26.7, o 30.9 / 28.8;
//     [20000,2688] 59.3 / 54.7, c 59.4 / 63.3, o 59.4 / 68.5).
inline bool nr_takes(bool bf16, bool layer, uint64_t rows, uint32_t cols, uint64_t cus) {
    if (cols <= 256 || cols > NR_MAX_COLS || rows > NR_MAX_ROWS) return false;
    if (!layer) {
        if (bf16 || rows <= 16 * cus) return true;
        const uint32_t nt = (cols + 255) / 256;
        const bool lines = cols % 32 == 0;                   // rows start on 64 bytes
        if (cols >= 3072) return rows > 28 * cus && (!lines || nt != nf_steps(nt) || (cols > 4864 && rows > 30 * cus));
        return cols >= 320 && rows > (!lines || cols <= 512 ? 48 : 60) * cus;
    }
    if (!bf16) {
        if (cols <= 448) return rows <= 4 * cus;
        return rows <= cus / 16 || (cols <= 3584 && rows <= (cols <= 768 ? cus / 2 : cus));
    }
    if (rows <= 4 * cus) return true;
    if (rows <= 11 * cus) return cols <= 3072;
    if (rows > 16 * cus && rows <= 24 * cus) return cols > 768 && cols <= 1024;
    if (cols > 1024 && cols <= 1536) return rows > 32 * cus;
    return cols > 2048 && cols <= 2560 && rows > 30 * cus && rows <= 64 * cus;
}
// Where norm_flow16_kernel takes the rest of them, against norm_pipe16_kernel, whose blocks of 8 rows share the CUs and overlap one another,
// while rows fit the chip in a few rounds, and which needs no empty steps.  Many rows come to memory, which that one
// reads twice (LayerNorm f16 [12288,1024] 16.4 / 12.2, [24000,2560] 62 / 51).  Up to 40 rows a CU, f16 gains on rows of more than 3072 columns
// that fill the steps (RMSNorm [7000,4096] 27.8 / 23.5, against [5000,3328] 17.6 / 18.9).  bf16 LayerNorm, whose walker
// needs the f32 tiles of both sums, gains in a single round of 8 rows a block (measured at [2048,2560] 16.3 / 14.6, which the wave per row now takes)
// and once its blocks of 8 rows no longer keep their rows in LDS ([7000,2560] 35 / 25.6; [5000,2560] 21.3 / 25.8), except for short rows and for 9000 to 10000 rows in steps a quarter empty ([9000,1792] 29.4 / 27.9).
inline bool nf_takes_aligned(bool bf16, bool layer, uint64_t rows, uint32_t cols, uint64_t cus) {
    const uint32_t nt = (cols + 255) / 256, steps = nf_steps(nt);
    if (bf16 && layer) {
        if (rows <= 8 * cus) return cols > 3072;
        if (rows <= 16 * cus) return cols > 3328;
        if (rows <= 24 * cus || cols <= 128) return false;
        if (cols <= 256) return rows > 48 * cus;
        if (rows <= 32 * cus || rows > 42 * cus) return true;
        return nt * 5 >= steps * 4;
    }
    if (rows > 40 * cus) return cols > 512;                  // (RMSNorm in bf16: rows beyond NR_MAX_ROWS)
    if (bf16 || cols <= 3072) return false;
    if (nt == steps) return layer || rows > 8 * cus;
    return layer && rows >= 64 && rows <= 16 * cus && cols > 3328;
}

template <typename T, int KIND, int RB>
int launch_norm16_flow(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols, float eps) {
    // one block per CU; the groups as even as they can be over the fewest rounds
    const uint64_t cus = (uint64_t)dev->num_cus, rounds = (rows + cus * RB - 1) / (cus * RB);
    const uint32_t R = (uint32_t)((rows + cus * rounds - 1) / (cus * rounds));
    const uint64_t groups = (rows + R - 1) / R;
    RT_REQUIRE(groups <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
    // the walker and a loader wave for every two of the R <= RB rows: waves without a row would issue every instruction of the
    // others ([16384,3072], 64 rows a CU in rounds of 22: LayerNorm bf16 55.1 -> 48.1 us, f16 45.3 -> 43.0, RMSNorm bf16 43.7 -> 40.8).
    // Blocks of 8 rows launch all four: they stage the weights together, where one wave, for one or two rows, takes a trip for every 512
    // columns (LayerNorm f16 [1,4096] 16.7 us, 15.7 with four, [64,1001] 6.85 / 6.65)
    const uint32_t threads = 64 + (RB == 8 ? 4 : (R + 1) / 2) * 64;
    const uint32_t nt = (cols + 255) / 256;
    const size_t affine_bytes = (size_t)nt * 512 * (KIND == NORM_LAYER ? 2 : 1);
    const uint32_t steps = nf_steps(nt);
#define RT_FLOW(NT)                                                                                                                  \
    hipLaunchKernelGGL((norm_flow16_kernel<T, KIND, NT, RB>), dim3((unsigned)(groups < cus ? groups : cus)), dim3(threads),          \
                       affine_bytes, dev->stream, (const T*)x, (const T*)scale, (const T*)bias, (T*)y, rows, cols, (uint32_t)groups, R, eps)
    if (steps == 2) RT_FLOW(2);
    else if (steps == 4) RT_FLOW(4);
    else if (steps == 8) RT_FLOW(8);
    else if (steps == 12) RT_FLOW(12);
    else if (steps == 16) RT_FLOW(16);
    else RT_FLOW(20);
#undef RT_FLOW
    RT_CHECK_LAUNCH("norm_flow16_kernel");
    return RT_OK;
}

// the row walk is latency bound, so prefer many small row groups until the chip is covered a few times over
template <typename T, int KIND>
int launch_norm16(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols, float eps) {
    const bool vec_ok = (cols % 8 == 0) && rt_aligned(x, 16) && rt_aligned(y, 16) && rt_aligned(scale, 16) && (!bias || rt_aligned(bias, 16));
    if (vec_ok && cols <= 128 && rows >= 16384) return launch_norm16_lane<T, KIND>(dev, x, scale, bias, y, rows, cols, eps);
    const uint64_t cus = (uint64_t)dev->num_cus;
    constexpr bool BF16 = std::is_same<T, bf16_t>::value, LAYER = KIND == NORM_LAYER;
    if (vec_ok && nr_takes(BF16, LAYER, rows, cols, cus)) return rt_norm16_row(dev, BF16, KIND, x, scale, bias, y, rows, cols, eps);
    if (cols >= 8 && cols <= NF_MAX_COLS &&
        (vec_ok ? nf_takes_aligned(BF16, LAYER, rows, cols, cus) : nf_takes_ragged(BF16, LAYER, rows, cols, cus))) {
        // rows a block walks at one time: 30 fill its 1024 threads and the walker's lanes; fewer where that takes no more
        // rounds (a walk costs the same for any number of rows: RMSNorm f16 [5000,4096] 27 us in two rounds of 16, 21 in one of
        // 30).  LayerNorm rows of 20 steps: three rounds of 16 rather than two of 30, which spill ([10240,5113] f16 56 / 62)
        if (rows <= 8 * cus) return launch_norm16_flow<T, KIND, 8>(dev, x, scale, bias, y, rows, cols, eps);
        if (rows <= 16 * cus || (rows > 30 * cus && rows <= (LAYER && cols > 4096 ? 40 : 32) * cus))
            return launch_norm16_flow<T, KIND, 16>(dev, x, scale, bias, y, rows, cols, eps);
        return launch_norm16_flow<T, KIND, 30>(dev, x, scale, bias, y, rows, cols, eps);
    }
    if (vec_ok) {
        const uint64_t blocks = (rows + 7) / 8;
        RT_REQUIRE(blocks <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
        // all blocks resident at once (the latency-bound case): the output pass comes from LDS
        const uint32_t ntiles = (cols + 255) / 256;
        const size_t keep_bytes = (size_t)ntiles * NP_KEEP_BYTES_PER_TILE;
        const size_t static_bytes = (KIND == NORM_LAYER ? 2 : 1) * 2 * 8 * (std::is_same<T, half_t>::value ? 264 * 2 : 260 * sizeof(float)) + 256;
        const size_t per_cu = (160 * 1024) / (static_bytes + keep_bytes);
        if (cols <= NP_KEEP_MAX_COLS && blocks <= (uint64_t)dev->num_cus * per_cu) {
            const int ti = (std::is_same<T, half_t>::value ? 0 : 2) + (KIND == NORM_LAYER ? 0 : 1);
            if (!(dev->np_attr_set & (1u << ti))) {
                RT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(norm_pipe16_kernel<T, KIND, true>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)((NP_KEEP_MAX_COLS / 256) * NP_KEEP_BYTES_PER_TILE)));
                dev->np_attr_set |= 1u << ti;
            }
            hipLaunchKernelGGL((norm_pipe16_kernel<T, KIND, true>), dim3((unsigned)blocks), dim3(NP_BLOCK), keep_bytes, dev->stream, (const T*)x,
                               (const T*)scale, (const T*)bias, (T*)y, rows, cols, eps);
        } else {
            hipLaunchKernelGGL((norm_pipe16_kernel<T, KIND, false>), dim3((unsigned)blocks), dim3(NP_BLOCK), 0, dev->stream, (const T*)x,
                               (const T*)scale, (const T*)bias, (T*)y, rows, cols, eps);
        }
        RT_CHECK_LAUNCH("norm_pipe16_kernel");
        return RT_OK;
    }
    const uint64_t want_blocks = (uint64_t)dev->num_cus * 4;
    if (rows / 32 >= want_blocks) return launch_norm16_rb<T, KIND, 32>(dev, x, scale, bias, y, rows, cols, eps);
    if (rows / 16 >= want_blocks) return launch_norm16_rb<T, KIND, 16>(dev, x, scale, bias, y, rows, cols, eps);
    return launch_norm16_rb<T, KIND, 8>(dev, x, scale, bias, y, rows, cols, eps);
}

int norm_entry(rt_device* dev, int kind, int dt, const void* x, const void* scale, const void* bias, void* y, uint64_t rows,
               uint32_t cols, float eps, const char* who) {
    RT_REQUIRE(rt_is_float_dt(dt), RT_ERR_DTYPE, "%s: dtype %d is not F32/F16/BF16", who, dt);
    RT_REQUIRE(cols > 0, RT_ERR_SHAPE, "%s: cols is 0", who);
    RT_REQUIRE(rows <= RT_MAX_NUMEL / cols, RT_ERR_SIZE, "%s: tensor too large", who);
    RT_REQUIRE(eps == eps, RT_ERR_ARG, "%s: eps is NaN", who);
    if (rows == 0) return dev ? RT_OK : rt_fail(RT_ERR_NULL_DEVICE, "rt_device is NULL");
    RT_REQUIRE(x && scale && y, RT_ERR_NULL_POINTER, "%s: NULL operand", who);
    const size_t eb = (size_t)rt_dt_bytes(dt);
    RT_REQUIRE(rt_aligned(x, eb) && rt_aligned(y, eb) && rt_aligned(scale, eb) && (!bias || rt_aligned(bias, eb)), RT_ERR_ALIGN,
               "%s: misaligned pointer", who);
    int rc = rt_enter(dev);
    if (rc) return rc;
    if (kind == NORM_LAYER) {
        switch (dt) {
            case RT_F32: return launch_norm<float, NORM_LAYER>(dev, x, scale, bias, y, rows, cols, eps);
            case RT_F16: return launch_norm16<half_t, NORM_LAYER>(dev, x, scale, bias, y, rows, cols, eps);
            default: return launch_norm16<bf16_t, NORM_LAYER>(dev, x, scale, bias, y, rows, cols, eps);
        }
    }
    switch (dt) {
        case RT_F32: return launch_norm<float, NORM_RMS>(dev, x, scale, nullptr, y, rows, cols, eps);
        case RT_F16: return launch_norm16<half_t, NORM_RMS>(dev, x, scale, nullptr, y, rows, cols, eps);
        default: return launch_norm16<bf16_t, NORM_RMS>(dev, x, scale, nullptr, y, rows, cols, eps);
    }
}

// the threads' sums of a block, added in double: at the size of a whole group's sum each of these additions would cost half an ulp of it.
// `red` is the call's own: a second call may write while a wave still reads for the first
template <int BT> __device__ __forceinline__ double gn_block_sum(float v, double (&red)[BT / WAVE]) {
    const double sum = wave_sum((double)v);
    if ((threadIdx.x & (WAVE - 1)) == 0) red[threadIdx.x / WAVE] = sum;
    __syncthreads();
    constexpr int N = BT / WAVE;                             // 4, 8 or 16 sums, repeated over the lanes: the same butterfly in every wave
    double t = red[threadIdx.x & (N - 1)];
    if constexpr (N == 16) t = wave_step_sum<8>(t);
    if constexpr (N >= 8) t = wave_step_sum<4>(t);
    t = wave_step_sum<2>(t);
    return wave_step_sum<1>(t);
}

// 1 / sqrt(v) in double, as the launches for larger groups compute it: the total of the squares of a group, its quotient and a variance
// below f32's normal range stay representable (f32 [8,320,4097] of deviation 1.2e17 has a total of 5.8e38, which is inf in f32).  The
// instruction's estimate is good to about 2^-23, one step makes that 2^-45; where the step means nothing (v of 0 or inf) it is left out.
__device__ __forceinline__ float gn_rstd(double v) {
    const double r = __builtin_amdgcn_rsq(v), e = __builtin_fma(-v * r, r, 1.0);
    return (float)(__builtin_fabs(e) < 0.5 ? __builtin_fma(0.5 * r, e, r) : r);
}

// GroupNorm in one launch: the group in the registers of one block (thread t of BT holds vectors t, t + BT, ...; NV of them), so
// HBM sees it once; mean, squared deviations and the output are computed from the registers, with the definitions of the two-kernel
// path (mean, then the variance about that mean, f32 arithmetic).  What bounds it is how much of a CU's loads, reductions and
// stores run at the same time: WPE is the number of waves per SIMD that the registers leave room for, and with the sizes that
// launch_gn takes two blocks or more share a CU, one storing while another loads ([16,512,3000] f16, 512 groups of 94 KiB: 22.6 us with the
// group in LDS, one block to a CU, 20.3 with 1024 threads of 6 vectors, 20.4 with 512 of 12; [128,256,3000] f16 97 -> 63 us = 6.2 TB/s;
// [64,256,1500] f32 35.3 -> 30.0 us).
// SPAN: groups that do not start or end on a vector boundary, over the aligned vectors that cover them.  The elements of the
// neighbouring groups in the first and the last of those stay out of the sums and are not written (such vectors are stored element
// by element); an aligned vector that holds one byte of the tensor lies in a mapped page.  [16,320,3001] f16 55 -> 15 us against
// the element-wise launches.
// Few groups (fewer than half as many as CUs): `slices` blocks per group, all in one launch and without any wait between blocks.  Every
// block of a group loads the WHOLE group and reduces it to the same mean and variance in the same order, so the blocks of a
// group agree bit for bit without exchanging anything; each then normalises and stores only its own run of nvec / slices
// vectors.  The repeated reads of a group hit the L2 of the XCD its blocks share (see launch_gn_reg).
template <typename T, int NV, int BT, int WPE, bool SPAN>
__global__ void __launch_bounds__(BT, WPE) gn_reg_kernel(const T* __restrict__ x, const T* __restrict__ scale, const T* __restrict__ bias,
                                                         T* __restrict__ y, uint32_t glen, double inv_n, uint32_t cpg, uint32_t groups, FastDiv L,
                                                         float eps, uint32_t slices, uint32_t per_xcd) {
    constexpr int VE = 16 / sizeof(T);                       // inv_n: 1 / glen
    // blocks are handed to the 8 XCDs round robin: pair index p runs over the (group, slice) pairs of one XCD first
    const uint32_t p = per_xcd ? (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3) : blockIdx.x;
    const uint32_t grp = p / slices, slice = p - grp * slices, g = grp % groups;
    const uint64_t first = (uint64_t)grp * glen;
    const uint32_t shift = SPAN ? (uint32_t)(first & (VE - 1)) : 0;
    const v4u* xs = reinterpret_cast<const v4u*>(x) + first / VE;
    v4u* ys = reinterpret_cast<v4u*>(y) + first / VE;
    const uint32_t nvec = SPAN ? (shift + glen + VE - 1) / VE : glen / VE;
    auto ragged = [&](uint32_t i) -> bool { return SPAN && i < nvec && (i == 0 || i == nvec - 1); };
    auto inside = [&](uint32_t i, int q) -> bool { return i * VE + (uint32_t)q - shift < glen; };
    Vec16<T> v[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = threadIdx.x + k * BT;
        v[k].u = v4u{0u, 0u, 0u, 0u};
        if (i < nvec) v[k].u = slices > 1 ? xs[i] : ld_stream(xs + i);
    }
    float acc = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = threadIdx.x + k * BT;
        if (ragged(i)) {
#pragma unroll
            for (int q = 0; q < VE; q++)
                if (inside(i, q)) acc = gn_plus<T>(v[k].e[q], acc);
        } else {
#pragma unroll
            for (int q = 0; q < VE; q++) acc = gn_plus<T>(v[k].e[q], acc);       // vectors past the group hold zeros
        }
    }
    // joined and divided in f32 the mean would be off by some ulps, which all outputs of the group share: f32 [8,320,4097] of
    // mean 100 and deviation 1 was 5.6e-6 from 64 bits, is now 2.2e-6 (the launches for larger groups: 2.5e-6)
    __shared__ double red[2][BT / WAVE];
    const float mean = (float)(gn_block_sum<BT>(acc, red[0]) * inv_n);
    // the group stays in registers as it was loaded: the widened values of one pass must not be kept for the next, but with few
    // blocks of few vectors, which run alone on their CU and where keeping what fits saves instructions (32 groups of 93 KiB f16
    // 6.0 us, 6.8 when every pass widens again)
    constexpr bool KEEP = sizeof(T) == 4 || (WPE <= 4 && NV <= 9);
    auto forget = [&]() {
#pragma unroll
        for (int k = 0; k < NV; k++) asm volatile("" : "+v"(v[k].u[0]), "+v"(v[k].u[1]), "+v"(v[k].u[2]), "+v"(v[k].u[3]));
    };
    if (!KEEP) forget();
    float m2 = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = threadIdx.x + k * BT;
        if (ragged(i)) {
#pragma unroll
            for (int q = 0; q < VE; q++)
                if (inside(i, q)) m2 = gn_dev2<T>(v[k].e[q], mean, m2);
        } else if (i < nvec) {
#pragma unroll
            for (int q = 0; q < VE; q++) m2 = gn_dev2<T>(v[k].e[q], mean, m2);
        }
    }
    const float rstd = gn_rstd(gn_block_sum<BT>(m2, red[1]) * inv_n + (double)eps);
    if (!KEEP) forget();
    const uint32_t lo = (uint32_t)(((uint64_t)nvec * slice) / slices), hi = (uint32_t)(((uint64_t)nvec * (slice + 1)) / slices);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const uint32_t i = threadIdx.x + k * BT;
        if (i < lo || i >= hi) continue;
        if (ragged(i)) {
            T* yg = y + first;
#pragma unroll
            for (int q = 0; q < VE; q++) {
                const uint32_t e = i * VE + (uint32_t)q - shift;
                if (e < glen) {
                    const uint32_t c = g * cpg + fd_div(e, L);
                    const float w = scale ? Ar<T>::widen(scale[c]) : 1.0f, b = bias ? Ar<T>::widen(bias[c]) : 0.0f;
                    yg[e] = Ar<T>::conv(__builtin_fmaf(gn_plus<T>(v[k].e[q], -mean) * rstd, w, b));
                }
            }
        } else {
            st_stream(ys + i, gn_affine_vec<T>(v[k], i * VE - shift, g * cpg, L, scale, bias, mean, rstd));
        }
    }
}

// Many slices per group (few, very large groups): the partials of a group are combined once, by one block, into a
// single (mean, M2, count) triple that the apply kernel then reads as if the group had one slice.
__global__ void __launch_bounds__(BLOCK) gn_combine_kernel(const float* __restrict__ part, float* __restrict__ out, uint32_t splits) {
    __shared__ double s_n[BLOCK], s_mean[BLOCK], s_m2[BLOCK];
    const float* p = part + (uint64_t)blockIdx.x * splits * 3;
    double n = 0.0, mean = 0.0, m2 = 0.0;
    auto merge = [&](double nb, double mb, double m2b) {                       // Chan et al.
        if (nb == 0.0) return;
        const double nt = n + nb;
        const double delta = mb - mean;
        mean += delta * (nb / nt);
        m2 += m2b + delta * delta * (n * nb / nt);
        n = nt;
    };
    for (uint32_t k = threadIdx.x; k < splits; k += BLOCK) merge((double)p[3 * k + 2], (double)p[3 * k], (double)p[3 * k + 1]);
    s_n[threadIdx.x] = n;
    s_mean[threadIdx.x] = mean;
    s_m2[threadIdx.x] = m2;
    __syncthreads();
    for (int off = BLOCK / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            merge(s_n[threadIdx.x + off], s_mean[threadIdx.x + off], s_m2[threadIdx.x + off]);
            s_n[threadIdx.x] = n;
            s_mean[threadIdx.x] = mean;
            s_m2[threadIdx.x] = m2;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        float* o = out + (uint64_t)blockIdx.x * 3;
        o[0] = (float)mean;
        o[1] = (float)m2;
        o[2] = (float)n;
    }
}

template <typename T, int NV, int BT, int WPE, bool SPAN>
int launch_gn_reg(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint32_t bg, uint32_t glen, uint32_t cpg,
                  uint32_t groups, uint32_t L, float eps, uint32_t slices) {
    // with a block count that the 8 XCDs share evenly, block b (on XCD b % 8) takes pair (b % 8) * blocks / 8 + b / 8, which
    // puts the slices of a group on one XCD (all of them when bg is a multiple of 8)
    const uint32_t blocks = bg * slices, per_xcd = (slices > 1 && blocks % 8 == 0) ? blocks / 8 : 0;
    hipLaunchKernelGGL((gn_reg_kernel<T, NV, BT, WPE, SPAN>), dim3(blocks), dim3(BT), 0, dev->stream, (const T*)x, (const T*)scale, (const T*)bias,
                       (T*)y, glen, 1.0 / (double)glen, cpg, groups, make_fastdiv(L), eps, slices, per_xcd);
    RT_CHECK_LAUNCH("gn_reg_kernel");
    return RT_OK;
}

// fixed_scratch == nullptr: partial statistics go to the device's own buffer, grown from the driver when a problem needs
// more; otherwise to fixed_scratch (GN_STATIC_SCRATCH_BYTES), and a problem that needs more is refused.
template <typename T>
int launch_gn(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint32_t bg, uint32_t glen, uint32_t cpg,
              uint32_t groups, uint32_t L, float eps, float* fixed_scratch) {
    // enough blocks to cover the chip, slices of at least 2048 elements; beyond 64 slices per group the partials are
    // combined by a launch of their own instead of by every apply block
    constexpr uint32_t FUSED_COMBINE_MAX = 64;
    static_assert(FUSED_COMBINE_MAX <= WAVE, "gn_apply_kernel combines one partial per lane of a wave");
    uint32_t splits = (2048 + bg - 1) / bg;
    const uint32_t max_splits = (glen + 2047) / 2048;
    if (splits > max_splits) splits = max_splits;
    if (splits > 2048) splits = 2048;
    if (splits < 1) splits = 1;
    constexpr int VEMAX = 16 / sizeof(T);
    const bool aligned = rt_aligned(x, 16) && rt_aligned(y, 16);
    const bool vec = (glen % VEMAX == 0) && aligned;    // every group starts on a vector boundary
    // slices of at most 32 KiB stay in the registers of their 256-thread block (8 vectors a thread), in the stats launch and
    // in the apply launch: more, smaller slices when the rule above leaves them larger
    constexpr uint32_t GN_SLICE_REG_VEC = 8;
    constexpr uint32_t slice_reg_elems = GN_SLICE_REG_VEC * BLOCK * VEMAX;
    if (vec) {
        const uint32_t want = (glen + slice_reg_elems - 1) / slice_reg_elems;
        // (only while the partials still fit the fixed buffer of rt_group_norm_static: both entry points slice alike)
        if (want > splits && want <= 2048 && ((size_t)bg * want + bg) * 3 * sizeof(float) <= GN_STATIC_SCRATCH_BYTES) splits = want;
    }
    uint32_t chunk = (glen + splits - 1) / splits;
    if (vec) chunk = (chunk + VEMAX - 1) / VEMAX * VEMAX;                               // slices start on vector boundaries
    splits = (glen + chunk - 1) / chunk;
    const bool slice_reg = vec && chunk <= slice_reg_elems;
    const uint32_t slice_nv = slice_reg ? (chunk / VEMAX + BLOCK - 1) / BLOCK : 0;
    const size_t need = ((size_t)bg * splits + bg) * 3 * sizeof(float);           // partials, then one combined triple per group
    if (fixed_scratch)                                                              // whichever path the problem then takes
        RT_REQUIRE(need <= GN_STATIC_SCRATCH_BYTES, RT_ERR_SIZE,
                   "rt_group_norm_static: %u (batch, group) pairs in %u slices need %zu bytes of partial statistics, the fixed buffer holds %zu",
                   bg, splits, need, GN_STATIC_SCRATCH_BYTES);
    // Which path (measured on 256 CUs, us against the launches below or the next kernel that would hold the group):
    //   at most half as many groups as CUs, up to 144 KiB (192 in f32): 1024 threads, cus / groups blocks per group (32 groups of
    //        93 KiB f16 5.8, 6.9 by launches; ragged [2,320,3001] f16 7.9 / 10.7).  Larger ones in 16 bits go to the launches (64 groups
    //        of 160 KiB f16 13.3 / 9.6).  In place only one block a group may work (the others would load what it has stored), the launches
    //        keep the chip: theirs are long groups, up to a quarter as many as CUs (f16, one block / launches: 94 KiB x 32 groups 7.5 / 6.2,
    //        x 64 8.0 / 7.8, x 80 8.3 / 8.4, 144 KiB x 8 9.1 / 5.7; 50 KiB x 8 5.5 / 5.4, x 64 5.9 / 6.4; f32 120 KiB x 8 6.5 / 5.6)
    //   more groups: one block per group, as many threads as leave two blocks or more to a CU.  Up to 12, 24 and 48 KiB: 256, 512,
    //        512 threads of at most 3, 3, 6 vectors (8 KiB x 512 groups 5.0, 5.5 - 6.1 with wider blocks; 47 KiB x 2048 33.8, 35.7
    //        with 1024 threads); up to 96 KiB: 1024 threads of 4 or 6 (94 KiB x 256 groups 9.9, 11.5 with 512 threads of 12); up to
    //        128 KiB 512 threads of 16, which leave room for a second block where 1024 of 8 spill (125 KiB f32 x 512 21.2 / 26.6), but in
    //        16 bits only where there is a second block: up to one group a CU 1024 threads of 9 convert faster (127 KiB f16 x 129
    //        10.4 / 15.9, x 256 13.2 / 17.4; f32 x 256 12.6 / 12.3); up to 192 KiB 1024 threads of 9 or 12, one block to a CU
    //        (141 KiB f16 x 512 31.7, 39.4 by launches; 188 KiB f16 x 512 39.5 / 46.8).  16-bit groups of 12 vectors a thread are bound by
    //        their conversions, so a last round that is nearly empty costs what a full one does, and the launches take those: fewer than
    //        9/16 of the CUs in the first round, 5/8 of all rounds later (f16, one block / launches: 190 KiB x 129 17.5 / 14.0, x 160
    //        18.1 / 16.7, 148 KiB x 129 13.3 / 13.0, x 160 13.0 / 13.2; 148 KiB x 257 28.6 / 21.0, x 300 29.8 / 25.5, x 341 30.3 / 27.7, 190
    //        KiB x 300 35.1 / 32.4, x 341 35.9 / 37.0; bf16 148 KiB x 144 11.7 / 11.8).  Ragged ones never do (the launches go by element)
    //   f32 groups of 192 to 256 KiB (16 vectors a thread; 20 and 24 spill), at least as many groups as CUs: 250 KiB x 512 43.6, 61.9
    //        by launches; 256 KiB x 128: 16.5 / 16.4.  In 16 bits such groups go to the launches (x 512 64.2, 65.8 with 16 vectors)
    //   everything else: the launches below
    const uint32_t cus = (uint32_t)dev->num_cus;
    const uint32_t nvec = vec ? glen / VEMAX : (glen + 2 * VEMAX - 2) / VEMAX;          // the most vectors a group touches
#define RT_GN_REG(NVC, BTC, WPEC)                                                                                                    \
    return vec ? launch_gn_reg<T, NVC, BTC, WPEC, false>(dev, x, scale, bias, y, bg, glen, cpg, groups, L, eps, slices)          \
               : launch_gn_reg<T, NVC, BTC, WPEC, true>(dev, x, scale, bias, y, bg, glen, cpg, groups, L, eps, slices)
    const bool spread_in_place = x == y && 4u * bg <= cus && glen > 26624 + 96 * bg;
    if (aligned && 2u * bg <= cus && nvec <= (sizeof(T) == 4 ? 12288u : 9216u) && !spread_in_place) {
        uint32_t slices = x == y ? 1 : cus / bg;                        // in place, a block must not store what another still loads
        if (slices > 32) slices = 32;
        if (slices > nvec) slices = nvec;
        if (nvec <= 1024) RT_GN_REG(1, 1024, 4);
        if (nvec <= 2048) RT_GN_REG(2, 1024, 4);
        if (nvec <= 4096) RT_GN_REG(4, 1024, 4);
        if (nvec <= 6144) RT_GN_REG(6, 1024, 4);
        if (nvec <= 9216) RT_GN_REG(9, 1024, 4);
        RT_GN_REG(12, 1024, 4);
    }
    if (aligned && 2u * bg > cus) {
        const uint32_t slices = 1;
        if (nvec <= 768) RT_GN_REG(3, 256, 8);
        if (nvec <= 1536) RT_GN_REG(3, 512, 8);
        if (nvec <= 3072) RT_GN_REG(6, 512, 8);
        if (nvec <= 4096) RT_GN_REG(4, 1024, 8);
        if (nvec <= 6144) RT_GN_REG(6, 1024, 8);
        if (nvec <= 8192 && (sizeof(T) == 4 || bg > cus)) RT_GN_REG(16, 512, 4);
        if (nvec <= 9216) RT_GN_REG(9, 1024, 4);
        const uint64_t rounds = ((uint64_t)bg + cus - 1) / cus, enough = rounds == 1 ? cus * 9 / 16 : rounds * cus * 5 / 8;
        if (nvec <= 12288 && (sizeof(T) == 4 || !vec || bg >= enough)) RT_GN_REG(12, 1024, 4);
        if constexpr (sizeof(T) == 4) {
            if (nvec <= 16384 && bg >= cus) RT_GN_REG(16, 1024, 4);
        }
    }
#undef RT_GN_REG
    if (!fixed_scratch && need > dev->gn_scratch_bytes) {
        RT_NO_CAPTURE(dev, "growing the GroupNorm scratch");
        RT_HIP(hipStreamSynchronize(dev->stream));
        RT_HIP(hipFree(dev->gn_scratch));
        dev->gn_scratch = nullptr;
        dev->gn_scratch_bytes = 0;
        RT_HIP(hipMalloc((void**)&dev->gn_scratch, need));
        dev->gn_scratch_bytes = need;
    }
    const dim3 grid(bg, splits), block(BLOCK);
    const bool separate = splits > FUSED_COMBINE_MAX;
    float* const part = fixed_scratch ? fixed_scratch : dev->gn_scratch;
    const float* stats = separate ? part + (size_t)bg * splits * 3 : part;
    const uint32_t stat_splits = separate ? 1 : splits;
#define RT_GN_STATS(NVC) \
    hipLaunchKernelGGL((gn_stats_reg_kernel<T, NVC>), grid, block, 0, dev->stream, (const T*)x, part, glen, chunk, splits)
    if (slice_reg && slice_nv <= 1) RT_GN_STATS(1);
    else if (slice_reg && slice_nv <= 2) RT_GN_STATS(2);
    else if (slice_reg && slice_nv <= 4) RT_GN_STATS(4);
    else if (slice_reg) RT_GN_STATS(8);
    else if (vec) hipLaunchKernelGGL((gn_stats_kernel<T, VEMAX>), grid, block, 0, dev->stream, (const T*)x, part, glen, chunk, splits);
    else hipLaunchKernelGGL((gn_stats_kernel<T, 1>), grid, block, 0, dev->stream, (const T*)x, part, glen, chunk, splits);
#undef RT_GN_STATS
    RT_CHECK_LAUNCH("gn_stats_kernel");
    if (separate) {
        hipLaunchKernelGGL(gn_combine_kernel, dim3(bg), block, 0, dev->stream, (const float*)part,
                           part + (size_t)bg * splits * 3, splits);
        RT_CHECK_LAUNCH("gn_combine_kernel");
    }
#define RT_GN_APPLY(NVC)                                                                                                                   \
    hipLaunchKernelGGL((gn_apply_reg_kernel<T, NVC>), grid, block, 0, dev->stream, (const T*)x, (const T*)scale, (const T*)bias, (T*)y, stats, \
                       glen, chunk, stat_splits, cpg, groups, make_fastdiv(L), eps)
    if (slice_reg && slice_nv <= 1) RT_GN_APPLY(1);
    else if (slice_reg && slice_nv <= 2) RT_GN_APPLY(2);
    else if (slice_reg && slice_nv <= 4) RT_GN_APPLY(4);
    else if (slice_reg) RT_GN_APPLY(8);
#undef RT_GN_APPLY
    else if (vec) {
        hipLaunchKernelGGL((gn_apply_kernel<T, VEMAX>), grid, block, 0, dev->stream, (const T*)x, (const T*)scale, (const T*)bias, (T*)y, stats,
                           glen, chunk, stat_splits, cpg, groups, make_fastdiv(L), eps);
    } else {
        hipLaunchKernelGGL((gn_apply_kernel<T, 1>), grid, block, 0, dev->stream, (const T*)x, (const T*)scale, (const T*)bias, (T*)y, stats,
                           glen, chunk, stat_splits, cpg, groups, make_fastdiv(L), eps);
    }
    RT_CHECK_LAUNCH("gn_apply_kernel");
    return RT_OK;
}

template <typename T, int KIND>
int launch_norm_via32(rt_device* dev, const void* x, const float* scale, const float* bias, void* y, uint64_t rows, uint32_t cols, float eps) {
    const uint32_t nvec = cols / 8;
    const bool vec_ok = (cols % 8 == 0) && rt_aligned(x, 16) && rt_aligned(y, 16) && rt_aligned(scale, 16) && (!bias || rt_aligned(bias, 16)) &&
                        nvec <= (uint32_t)(BLOCK * 8);
    if (vec_ok && nvec <= 32) {
        // rows of at most 32 vectors: a group of 2..32 lanes per row (one vector each), so that a wave carries 2..32 rows
        // and as many bytes as with long rows
        const uint32_t lanes = nvec <= 2 ? 2 : nvec <= 4 ? 4 : nvec <= 8 ? 8 : nvec <= 16 ? 16 : 32;
        const uint64_t blocks = (rows + BLOCK / lanes - 1) / (BLOCK / lanes);
        RT_REQUIRE(blocks <= 0x7fffffffull, RT_ERR_SIZE, "rt_norm_via_f32: too many rows");
        const dim3 grid((unsigned)blocks), block(BLOCK);
#define RT_NARROW(L) hipLaunchKernelGGL((norm_via32_wave_kernel<T, 1, KIND, L>), grid, block, 0, dev->stream, (const T*)x, scale, bias, (T*)y, rows, cols, eps)
        if (lanes == 2) RT_NARROW(2);
        else if (lanes == 4) RT_NARROW(4);
        else if (lanes == 8) RT_NARROW(8);
        else if (lanes == 16) RT_NARROW(16);
        else RT_NARROW(32);
#undef RT_NARROW
        RT_CHECK_LAUNCH("norm_via32_wave_kernel");
        return RT_OK;
    }
    if (vec_ok && nvec <= (uint32_t)(WAVE * 8)) {
        const uint32_t nv = (nvec + WAVE - 1) / WAVE;
        // LayerNorm over 16384 rows or more: a wave takes two rows and loads the weights once for both (measured against one
        // row a wave: [32768,2048] 49.5 against 51.8 us, [16384,3072] 39.2 against 41.9, [65536,512] 25.2 against 27.1; with fewer
        // rows the chip is not covered often enough for the fatter waves, [8192,4096] 30.5 against 28.8; four rows a wave
        // win on some shapes and lose on others; RMSNorm, with half the weights, gains nothing at any size)
        const int rw = KIND == NORM_LAYER && rows >= (uint64_t)dev->num_cus * 64 ? 2 : 1;
        const uint64_t blocks = ((rows + rw - 1) / rw + WAVES - 1) / WAVES;
        RT_REQUIRE(blocks <= 0x7fffffffull, RT_ERR_SIZE, "rt_norm_via_f32: too many rows");
        const dim3 grid((unsigned)blocks), block(BLOCK);
#define RT_NV(NVC, RWC) hipLaunchKernelGGL((norm_via32_rows_kernel<T, NVC, KIND, WAVE, RWC>), grid, block, 0, dev->stream, (const T*)x, scale, bias, (T*)y, rows, cols, eps)
#define RT_NV1(NVC) hipLaunchKernelGGL((norm_via32_wave_kernel<T, NVC, KIND, WAVE>), grid, block, 0, dev->stream, (const T*)x, scale, bias, (T*)y, rows, cols, eps)
#define RT_NV_RW2(NVC)               \
    do {                             \
        if (rw == 2) RT_NV(NVC, 2);  \
        else RT_NV1(NVC);            \
    } while (0)
        if (nv <= 1) RT_NV_RW2(1);
        else if (nv <= 2) RT_NV_RW2(2);
        else if (nv <= 4) RT_NV_RW2(4);
        else if (nv <= 6) RT_NV_RW2(6);
        else RT_NV_RW2(8);
#undef RT_NV_RW2
#undef RT_NV1
#undef RT_NV
        RT_CHECK_LAUNCH("norm_via32_wave_kernel");
        return RT_OK;
    }
    if (vec_ok) {
        const uint32_t nv = (nvec + BLOCK - 1) / BLOCK;
        RT_REQUIRE(rows <= 0x7fffffffull, RT_ERR_SIZE, "rt_norm_via_f32: too many rows");
        // LayerNorm over 2048 rows or more: a block takes two rows and loads the weights once for both ([2048,8192] 12.7 against
        // 17.2 us, [8192,5120] 35.5 against 38.5, [16384,8192] 99 against 115; RMSNorm gains nothing)
        const int rw = KIND == NORM_LAYER && rows >= (uint64_t)dev->num_cus * 8 ? 2 : 1;
        const dim3 grid((unsigned)((rows + rw - 1) / rw)), block(BLOCK);
#define RT_NV(NVC, RWC) hipLaunchKernelGGL((norm_via32_rows_kernel<T, NVC, KIND, BLOCK, RWC>), grid, block, 0, dev->stream, (const T*)x, scale, bias, (T*)y, rows, cols, eps)
#define RT_NV1(NVC) hipLaunchKernelGGL((norm_via32_wave_kernel<T, NVC, KIND, BLOCK>), grid, block, 0, dev->stream, (const T*)x, scale, bias, (T*)y, rows, cols, eps)
#define RT_NV_RW2(NVC)               \
    do {                             \
        if (rw == 2) RT_NV(NVC, 2);  \
        else RT_NV1(NVC);            \
    } while (0)
        if (nv <= 3) RT_NV_RW2(3);
        else if (nv <= 4) RT_NV_RW2(4);
        else if (nv <= 6) RT_NV_RW2(6);
        else RT_NV_RW2(8);
#undef RT_NV_RW2
#undef RT_NV1
#undef RT_NV
        RT_CHECK_LAUNCH("norm_via32_wave_kernel");
        return RT_OK;
    }
    RT_REQUIRE(rows <= 0x7fffffffull, RT_ERR_SIZE, "rt_norm_via_f32: too many rows");
    hipLaunchKernelGGL((norm_via32_generic_kernel<T, KIND>), dim3((unsigned)rows), dim3(BLOCK), 0, dev->stream, (const T*)x, scale, bias,
                       (T*)y, rows, cols, eps);
    RT_CHECK_LAUNCH("norm_via32_generic_kernel");
    return RT_OK;
}

}  // namespace

// Called by rt_device_create with the new device current: looks up where THIS device's copy of gn_static_scratch lies.
int rt_norm_device_init(rt_device* dev) {
    void* p = nullptr;
    RT_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(gn_static_scratch)));
    dev->gn_static_ptr = static_cast<float*>(p);
    return RT_OK;
}

extern "C" {

int rt_norm_via_f32(rt_device* dev, int kind, int io_dt, const void* x, const float* scale, const float* bias, void* y, uint64_t rows,
                    uint32_t cols, float eps) {
    RT_REQUIRE(kind == NORM_LAYER || kind == NORM_RMS, RT_ERR_ARG, "rt_norm_via_f32: kind %d is not 0 (layer) or 1 (rms)", kind);
    RT_REQUIRE(io_dt == RT_F16 || io_dt == RT_BF16, RT_ERR_DTYPE, "rt_norm_via_f32: dtype %d is not F16/BF16", io_dt);
    RT_REQUIRE(cols > 0, RT_ERR_SHAPE, "rt_norm_via_f32: cols is 0");
    RT_REQUIRE(rows <= RT_MAX_NUMEL / cols, RT_ERR_SIZE, "rt_norm_via_f32: tensor too large");
    RT_REQUIRE(eps == eps, RT_ERR_ARG, "rt_norm_via_f32: eps is NaN");
    if (rows == 0) return dev ? RT_OK : rt_fail(RT_ERR_NULL_DEVICE, "rt_device is NULL");
    RT_REQUIRE(x && scale && y, RT_ERR_NULL_POINTER, "rt_norm_via_f32: NULL operand");
    RT_REQUIRE(rt_aligned(x, 2) && rt_aligned(y, 2) && rt_aligned(scale, 4) && (!bias || rt_aligned(bias, 4)), RT_ERR_ALIGN,
               "rt_norm_via_f32: misaligned pointer");
    int rc = rt_enter(dev);
    if (rc) return rc;
    if (kind == NORM_RMS) bias = nullptr;
    if (io_dt == RT_F16)
        return kind == NORM_LAYER ? launch_norm_via32<half_t, NORM_LAYER>(dev, x, scale, bias, y, rows, cols, eps)
                                  : launch_norm_via32<half_t, NORM_RMS>(dev, x, scale, bias, y, rows, cols, eps);
    return kind == NORM_LAYER ? launch_norm_via32<bf16_t, NORM_LAYER>(dev, x, scale, bias, y, rows, cols, eps)
                              : launch_norm_via32<bf16_t, NORM_RMS>(dev, x, scale, bias, y, rows, cols, eps);
}

int rt_layer_norm(rt_device* dev, int dt, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols,
                  float eps) {
    return norm_entry(dev, NORM_LAYER, dt, x, scale, bias, y, rows, cols, eps, "rt_layer_norm");
}

int rt_rms_norm(rt_device* dev, int dt, const void* x, const void* scale, void* y, uint64_t rows, uint32_t cols, float eps) {
    return norm_entry(dev, NORM_RMS, dt, x, scale, nullptr, y, rows, cols, eps, "rt_rms_norm");
}

static int group_norm_entry(rt_device* dev, int dt, const void* x, const void* scale, const void* bias, void* y, uint32_t B, uint32_t C,
                            uint32_t L, uint32_t groups, float eps, bool fixed) {
    RT_REQUIRE(rt_is_float_dt(dt), RT_ERR_DTYPE, "rt_group_norm: dtype %d is not F32/F16/BF16", dt);
    RT_REQUIRE(B > 0 && C > 0 && L > 0, RT_ERR_SHAPE, "rt_group_norm: zero extent");
    RT_REQUIRE(groups > 0 && C % groups == 0, RT_ERR_ARG, "rt_group_norm: %u channels do not split into %u groups", C, groups);
    RT_REQUIRE(eps == eps, RT_ERR_ARG, "rt_group_norm: eps is NaN");
    const uint64_t glen = (uint64_t)(C / groups) * L;
    RT_REQUIRE(glen <= 0x7fffffffull && (uint64_t)B * groups <= 0x7fffffffull, RT_ERR_SIZE, "rt_group_norm: group too large");
    RT_REQUIRE(x && y, RT_ERR_NULL_POINTER, "rt_group_norm: NULL operand");
    const size_t eb = (size_t)rt_dt_bytes(dt);
    RT_REQUIRE(rt_aligned(x, eb) && rt_aligned(y, eb) && (!scale || rt_aligned(scale, eb)) && (!bias || rt_aligned(bias, eb)),
               RT_ERR_ALIGN, "rt_group_norm: misaligned pointer");
    int rc = rt_enter(dev);
    if (rc) return rc;
    const uint32_t bg = B * groups;
    float* fixed_scratch = nullptr;
    if (fixed) {
        fixed_scratch = dev->gn_static_ptr;
        RT_REQUIRE(fixed_scratch, RT_ERR_ARG, "rt_group_norm_static: the device's fixed scratch buffer was not resolved at rt_device_create");
    }
    switch (dt) {
        case RT_F32: return launch_gn<float>(dev, x, scale, bias, y, bg, (uint32_t)glen, C / groups, groups, L, eps, fixed_scratch);
        case RT_F16: return launch_gn<half_t>(dev, x, scale, bias, y, bg, (uint32_t)glen, C / groups, groups, L, eps, fixed_scratch);
        default: return launch_gn<bf16_t>(dev, x, scale, bias, y, bg, (uint32_t)glen, C / groups, groups, L, eps, fixed_scratch);
    }
}

int rt_group_norm(rt_device* dev, int dt, const void* x, const void* scale, const void* bias, void* y, uint32_t B, uint32_t C, uint32_t L,
                  uint32_t groups, float eps) {
    return group_norm_entry(dev, dt, x, scale, bias, y, B, C, L, groups, eps, false);
}

int rt_group_norm_static(rt_device* dev, int dt, const void* x, const void* scale, const void* bias, void* y, uint32_t B, uint32_t C,
                         uint32_t L, uint32_t groups, float eps) {
    return group_norm_entry(dev, dt, x, scale, bias, y, B, C, L, groups, eps, true);
}

}  // extern "C"
