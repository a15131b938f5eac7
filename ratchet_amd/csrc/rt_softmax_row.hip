// The 16-bit reference softmax, a wave per row, the row in registers: the left-to-right 16-bit sum of its exponentials without a walk
// (rt_ordered.h; arithmetic and table: rt_softmax_stream.h).
#include <cmath>

#include "rt_softmax_stream.h"
#include "rt_ordered.h"

namespace {

// The 16-bit chains of exponentials.  MANT: mantissa bits of the running sum's type, INF: its infinity's bit pattern.  pair(a, b) starts two sums at two bit
// patterns, run() adds a vector's eight terms to both, lo() and hi() are the sums' bit patterns; one() adds to a single sum.
template <typename T> struct Chain16;
template <> struct Chain16<half_t> {
    static constexpr int MANT = 10;
    static constexpr uint32_t INF = 0x7c00u;
    typedef uint32_t Pair;                                   // both sums in one register
    static __device__ __forceinline__ Pair pair(uint32_t a, uint32_t b) { return a | b << 16; }
    static __device__ __forceinline__ uint32_t lo(Pair p) { return p & 0xffffu; }
    static __device__ __forceinline__ uint32_t hi(Pair p) { return p >> 16; }
#define SR_LINK(N)                                                          \
    "v_pk_add_f16 %0, %0, %" #N " op_sel:[0,0] op_sel_hi:[1,0]\n"            \
    "v_pk_add_f16 %0, %0, %" #N " op_sel:[0,1] op_sel_hi:[1,1]\n"
    static __device__ __forceinline__ void run(Pair& p, const v4u& v) {
        asm(SR_LINK(1) SR_LINK(2) SR_LINK(3) SR_LINK(4) : "+v"(p) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
    }
#undef SR_LINK
    static __device__ __forceinline__ uint32_t one(uint32_t s, const v4u& v) {
        run(s, v);
        return s & 0xffffu;
    }
};
template <> struct Chain16<bf16_t> {
    static constexpr int MANT = 7;
    static constexpr uint32_t INF = 0x7f80u;
    struct Pair {
        uint32_t a, b;                                       // widened
    };
    static __device__ __forceinline__ Pair pair(uint32_t a, uint32_t b) { return Pair{a << 16, b << 16}; }
    static __device__ __forceinline__ uint32_t lo(const Pair& p) { return p.a >> 16; }
    static __device__ __forceinline__ uint32_t hi(const Pair& p) { return p.b >> 16; }
#define SR_ADD(A, X) "v_add_f32 " A ", " A ", " X "\n"
#define SR_ROUND(A) "v_cvt_pk_bf16_f32 " A ", 0, " A "\n"
#define SR_LINK(N)                                                                                                 \
    "v_lshlrev_b32 %2, 16, %" #N "\n" SR_ADD("%0", "%2") SR_ADD("%1", "%2") SR_ROUND("%0") SR_ROUND("%1")           \
    "v_and_b32 %2, 0xffff0000, %" #N "\n" SR_ADD("%0", "%2") SR_ADD("%1", "%2") SR_ROUND("%0") SR_ROUND("%1")
    static __device__ __forceinline__ void run(Pair& p, const v4u& v) {
        uint32_t t;
        asm(SR_LINK(3) SR_LINK(4) SR_LINK(5) SR_LINK(6) : "+v"(p.a), "+v"(p.b), "=&v"(t) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
    }
#undef SR_LINK
#define SR_LINK(N)                                                                     \
    "v_lshlrev_b32 %1, 16, %" #N "\n" SR_ADD("%0", "%1") SR_ROUND("%0")                 \
    "v_and_b32 %1, 0xffff0000, %" #N "\n" SR_ADD("%0", "%1") SR_ROUND("%0")
    static __device__ __forceinline__ uint32_t one(uint32_t s, const v4u& v) {
        uint32_t a = s << 16, t;
        asm(SR_LINK(2) SR_LINK(3) SR_LINK(4) SR_LINK(5) : "+v"(a), "=&v"(t) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
        return a >> 16;
    }
#undef SR_LINK
#undef SR_ROUND
#undef SR_ADD
};

// inclusive prefix sum over groups of L lanes (16 or 32)
template <int L> __device__ __forceinline__ uint32_t sr_scan(uint32_t v) {
    v += scan_move<0x111, 0xf>(v);                           // row_shr:1, 2, 4, 8
    v += scan_move<0x112, 0xf>(v);
    v += scan_move<0x114, 0xf>(v);
    v += scan_move<0x118, 0xf>(v);
    if (L == 32) v += scan_move<0x142, 0xa>(v);              // the last lane of rows 0 and 2 onto rows 1 and 3
    return v;
}

// A bit per group: its lowest, its highest lane
template <int L> constexpr uint64_t SR_LOW = L == 16 ? 0x0001000100010001ull : 0x0000000100000001ull;
template <int L> constexpr uint64_t SR_HIGH = SR_LOW<L> << (L - 1);

// The ordered sums (rt_ordered.h) of the 64 / L rows of a wave at one time: s, the bit pattern of a row's sum, is the same in the L lanes of its
// group; a lane has 32 terms.  A lane in which the sum leaves the binade adds for real in the same pass that prepares the lanes behind it for the next
// binade.  Nothing is approximated: a distance is used only if the sum stayed inside the binade it was made for (it never decreases, so every sum in
// between did too).  inf and NaN lie beyond every binade and are absorbed as the adder absorbs them.  All groups make the same passes, and those that are through idle: the passes that a row needs come
// mostly from the powers of two that its sum passes, which is at about the same columns in all of them.
template <class C, int L>
__device__ __forceinline__ uint32_t sr_group_add(uint32_t s, const v4u (&v)[4], uint32_t gl) {
    constexpr uint32_t ULPS = 1u << C::MANT;                 // sums in a binade
    const uint32_t group = (threadIdx.x & 63u) - gl;
    auto field_of = [&](uint64_t lanes) -> uint32_t {        // the group's lanes of a mask
        const uint32_t f = (uint32_t)(lanes >> group);
        return L == 16 ? f & 0xffffu : f;
    };
    uint32_t from = 0;                                       // lanes of the group below it are in s
    if (__builtin_amdgcn_ballot_w64(s == 0)) {               // at the start of a row the first lane adds for real
        uint32_t t = s;
#pragma unroll
        for (int k = 0; k < 4; k++) t = C::one(t, v[k]);
        t = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(group * 4), (int)t);
        if (s == 0) {
            s = t;
            from = 1;
        }
    }
    // inf stays, or some lane makes a NaN of it, which stays
    auto absorb = [&]() {
        const bool stuck = s >= C::INF;
        if (__builtin_amdgcn_ballot_w64(stuck) == 0) return;
        uint32_t t = s;
#pragma unroll
        for (int k = 0; k < 4; k++) t = C::one(t, v[k]);
        const uint64_t other = __builtin_amdgcn_ballot_w64(stuck & (gl >= from) & (t != s));
        if (field_of(other)) s = C::INF + ULPS / 2;
        if (stuck) from = L;
    };
    absorb();
    uint64_t real = 0;                                       // lanes that add to s itself: `from` of some groups
    // the binade that the lanes from `from` on prepare for; the subnormals and the first normal one have one ulp and count as one
    uint32_t base, size;
    auto binade = [&](uint32_t e) {
        base = e <= 1 ? 0 : e << C::MANT;
        size = e <= 1 ? 2 * ULPS : ULPS;
    };
    binade(s >> C::MANT);
    for (;;) {
        const bool mine = __builtin_amdgcn_inverse_ballot_w64(real), out = gl < from;
        const uint32_t at_first = mine ? s : base;
        typename C::Pair p = C::pair(at_first, base + 1);
#pragma unroll
        for (int k = 0; k < 4; k++) C::run(p, v[k]);
        const uint32_t lo = C::lo(p);
        uint32_t d0 = lo - at_first, d1 = C::hi(p) - (base + 1);
        if (mine) d1 = d0;
        if (out) d0 = d1 = 0;
        // the parity in front of each lane: `flips` is that of the distances before it alone, a tie (or a real sum) sets it anew
        const uint64_t outs = __builtin_amdgcn_ballot_w64(out);
        const uint64_t odd = __builtin_amdgcn_ballot_w64(lo & 1u) & ~outs, set = __builtin_amdgcn_ballot_w64(d0 != d1) | real;
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(odd >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)odd, 0));
        uint64_t flips = __builtin_amdgcn_ballot_w64(below & 1u);
        const uint64_t first = flips & SR_LOW<L>;            // (counted from the wave's first lane: from the group's on)
        flips ^= (first << L) - first;
        // prop + gen + in, carries stopping at a group's highest lane; what is wanted is the carry into each lane
        const uint64_t gen = set & flips, prop = gen | ~set, in = __builtin_amdgcn_ballot_w64(s & 1u) & SR_LOW<L>;
        const uint64_t a = prop & ~SR_HIGH<L>, b = gen & ~SR_HIGH<L>, parity = (a + b + in) ^ a ^ b ^ flips;
        const uint32_t d = __builtin_amdgcn_inverse_ballot_w64(parity) ? d1 : d0;
        const uint32_t upto = s + sr_scan<L>(d), before = upto - d;
        // a lane's distance holds if its run starts and ends in the binade
        const uint64_t bads = (__builtin_amdgcn_ballot_w64(before < base) | __builtin_amdgcn_ballot_w64(upto - base >= size)) & ~(outs | real);
        const uint32_t field = field_of(bads), at = field ? __builtin_ctz(field) : L;
        s = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((group + (at < L ? at : L - 1)) * 4),
                                                   (int)(__builtin_amdgcn_inverse_ballot_w64(bads) ? before : upto));
        if (bads == 0) return s;
        from = at;
        const bool there = s - base < size;                  // else the lanes behind the last one were prepared for another binade
        const uint32_t e = base >> C::MANT;
        absorb();
        binade(!there ? s >> C::MANT : e <= 1 ? 2 : e + 1);  // where the lanes behind that one most likely add
        real = __builtin_amdgcn_ballot_w64(there & (gl == from));
    }
}

// Four registers of a chunk in memory order, 64 lanes to 1 KiB of a row, become a lane's 32 consecutive terms in its row's group (register i
// before: L = 16: group i; L = 32: half i & 1 of the chunk of group i >> 1).  The register index and the two upper lane bits change places by
// swaps, and what that put into the register index goes to the place of the two lower lane bits by DPP moves, so a lane holds the vector
// before that sr_vector names: quads read 64 bytes, an instruction the whole KiB.  (Half of every line to an instruction, [1,8,700,6000] f16
// 49 us / 35 as here: rows start inside of lines, whose parts were written one by one.)
template <int CTRL> __device__ __forceinline__ uint32_t sr_quad(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, true);
}
template <int L> __device__ __forceinline__ uint32_t sr_vector(uint32_t lane, int i) {
    return (lane & 3) | (lane >> 4) << 2 | (lane >> 2 & 3) << 4 | (L == 32 ? (uint32_t)(i & 1) << 6 : 0);
}
__device__ __forceinline__ void sr_transpose(v4u (&v)[4], uint32_t lane) {
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const auto p = __builtin_amdgcn_permlane32_swap(v[0][w], v[2][w], false, false), q = __builtin_amdgcn_permlane32_swap(v[1][w], v[3][w], false, false);
        const auto r = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false), t = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
        v[0][w] = r[0];
        v[1][w] = r[1];
        v[2][w] = t[0];
        v[3][w] = t[1];
    }
    const bool odd = lane & 1, high = lane & 2;
#pragma unroll
    for (int k = 0; k < 4; k += 2)
#pragma unroll
        for (int w = 0; w < 4; w++) {
            // (the moves take part in every lane: not inside a conditional)
            const uint32_t a = v[k][w], b = v[k + 1][w], am = sr_quad<0xb1>(a), bm = sr_quad<0xb1>(b);      // quad_perm:[1,0,3,2]
            v[k][w] = odd ? bm : a;
            v[k + 1][w] = odd ? b : am;
        }
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const uint32_t a = v[k][w], b = v[k + 2][w], am = sr_quad<0x4e>(a), bm = sr_quad<0x4e>(b);      // quad_perm:[2,3,0,1]
            v[k][w] = high ? bm : a;
            v[k + 2][w] = high ? b : am;
        }
}

// ------------------------------------------------------------------------------------------------------------------
// A wave takes 64 / L rows: four of up to 2048 columns (L = 16 lanes to a row), two of up to 8192 (L = 32), held in registers from the load to the
// store, and its waves never meet: no walker, no barriers.  A chunk is 32 L columns of each row, four vectors a lane.  The loads of the next
// rows go out between the stores of these, into the registers that those free.  The exp table lies in LDS as in softmax16_stream_kernel.
// What bounds it: a tenth of the time is the sums and their waits (without them, and wrong, [8,2048,8192] f16 takes 100 us of 114, with a mask 114 of 125), the
// rest memory, which 16 free-running waves a CU use less evenly than the streaming kernel's paced steps do (5.3 against 6.2 TB/s on f16 [32,4096,4096], 407 and 344 us; held
// to a pace these waves only get slower).  Several rows at a time because a row needs a pass for each chunk and for each power of two that its
// sum passes, most of which fall together: with one row to a wave [8,2048,8192] bf16 took 159 us without a mask and 177 with one, now 124 and 139.
// bf16 pays five instructions an element and pass, f16 one.
// ------------------------------------------------------------------------------------------------------------------
constexpr uint32_t SR_NONE = 0x80000000u;                    // an offset outside every buffer, and so after adding a column's
constexpr int sr_waves(int v) { return v <= 4 ? 16 : v <= 6 ? 12 : 8; }

// Row i of the launch: with a mask the `reps` rows that share a mask row come one after the other, in the groups of a wave and then in neighbouring
// blocks, which read it at about the same time but on different XCDs: under eight heads two to a wave HBM is asked for it four times ([8,2048,8192] f16: 131 MiB
// of reads for a mask of 32 MiB, by FETCH_SIZE).
struct SrRows {
    uint32_t rows, cols, period, waves;                      // waves: of a block, that have rows
    FastDiv reps_div;                                        // reps = rows / period (1 without a mask)
};

template <typename T, int L, int V, bool MASK, bool RAGGED>
__global__ void __launch_bounds__(64 * sr_waves(V)) softmax16_row_kernel(const uint16_t* __restrict__ table, const T* x, const T* __restrict__ mask, T* y, SrRows g) {
    typedef SpType<T> ST;
    constexpr int BLOCK_T = 64 * sr_waves(V), R = 64 / L, M = 4 / R;         // M: vectors of a row in a chunk
    constexpr int LOADS = RAGGED ? 0 : 2;                    // (vectors across lines: the line stays for the next one; otherwise non-temporal)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), gl = lane & (L - 1);
    const uint32_t cols = g.cols, nvec = (cols + 7) / 8, row_bytes = cols * 2, dup = nvec * 8 - cols;
    const uint32_t total = g.rows * row_bytes;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(x), 0, total, 0x00020000);
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y, 0, total, 0x00020000);
    const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(MASK ? mask : x), 0, MASK ? g.period * row_bytes : total, 0x00020000);
    // the lane's vector of row `i * R / 4` of the wave's, in chunk j; its byte offset in a row that starts at `row`
    auto vector = [&](int j, int i) -> uint32_t { return j * 4 * L + sr_vector<L>(lane, i); };
    auto place = [&](uint32_t row, int j, int i) -> uint32_t {
        const uint32_t n = vector(j, i);
        if (j < V - 1) return row + n * 16;
        if (RAGGED && n == nvec - 1) return row + row_bytes - 16;
        return n < nvec ? row + n * 16 : SR_NONE;
    };
    struct Rows {
        uint32_t at[R];
    };
    auto rows_of = [&](uint32_t item, uint32_t& mrow) -> Rows {
        Rows r;
#pragma unroll
        for (int k = 0; k < R; k++) {
            const uint32_t i = item * R + k;
            uint32_t q = i, head = 0;
            if (MASK) fd_divmod(i, g.reps_div, q, head);
            if (k == 0) mrow = i < g.rows ? q * row_bytes : SR_NONE;         // (all of them: R divides reps)
            r.at[k] = i < g.rows ? (head * g.period + q) * row_bytes : SR_NONE;
        }
        return r;
    };
    const uint32_t items = (g.rows + R - 1) / R, stride = gridDim.x * g.waves;
    uint32_t it = wave < g.waves ? wave * gridDim.x + blockIdx.x : items;
    uint32_t mrow = 0;
    Rows row = rows_of(it, mrow);
    v4u v[V][4];
#pragma unroll
    for (int j = 0; j < V; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) {                        // as in the loop: as many accesses in flight on both ways into it
            __builtin_amdgcn_raw_buffer_store_b128(v4u{0, 0, 0, 0}, ry, SR_NONE, 0, 2);
            v[j][i] = __builtin_amdgcn_raw_buffer_load_b128(rx, place(row.at[i * R / 4], j, i), 0, LOADS);
        }
    {
        const v4u* src = reinterpret_cast<const v4u*>(table);
        v4u* dst = reinterpret_cast<v4u*>(smem);
#pragma unroll 4
        for (uint32_t i = threadIdx.x; i < SP_LUT_BYTES / 16; i += BLOCK_T) dst[i] = src[i];
    }
    __syncthreads();

#pragma unroll 1
    while (it < items) {
        v4u mk[M];
        if (MASK) {
#pragma unroll
            for (int i = 0; i < M; i++) mk[i] = __builtin_amdgcn_raw_buffer_load_b128(rm, place(mrow, 0, i), 0, 0);
        }
        uint32_t s = 0;
#pragma unroll
        for (int j = 0; j < V; j++) {
            v4u t[4];
            if (MASK) {
#pragma unroll
                for (int i = 0; i < 4; i++) v[j][i] = ST::add_vec(v[j][i], mk[i % M]);
#pragma unroll
                for (int i = 0; i < M; i++)
                    if (j + 1 < V) mk[i] = __builtin_amdgcn_raw_buffer_load_b128(rm, place(mrow, j + 1, i), 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v4u a = v[j][i];
#pragma unroll
                for (int w = 0; w < 4; w++) a[w] = sp_exp_lo(a[w]) | sp_exp_hi(a[w]) << 16;
                v[j][i] = t[i] = a;
                if (j == V - 1) {
                    // without the vectors past the row's end, and without what the last one repeats of the one before it
                    const uint32_t n = vector(j, i);
#pragma unroll
                    for (int w = 0; w < 4; w++) {
                        const uint32_t keep = dup > 2 * (uint32_t)w + 1 ? 0u : dup > 2 * (uint32_t)w ? 0xffff0000u : 0xffffffffu;
                        if (RAGGED && n == nvec - 1) t[i][w] &= keep;
                        if (n >= nvec) t[i][w] = 0;
                    }
                }
            }
            sr_transpose(t, lane);
            s = sr_group_add<Chain16<T>, L>(s, t, gl);
        }
        // (the values' widened forms of one use are not to be held for the next: they are twice the registers of the row)
        auto forget = [&]() {
#pragma unroll
            for (int j = 0; j < V; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) asm volatile("" : "+v"(v[j][i]));
        };
        forget();
        float sums[R], rinv[R], rlow[R], by[R];
        bool wide = false;                                   // a sum outside of the short division's range
#pragma unroll
        for (int k = 0; k < R; k++) {
            sums[k] = ST::widen_bits(__builtin_amdgcn_readlane(s, k * L));
            by[k] = 1.0f;
            if constexpr (std::is_same<T, bf16_t>::value) {  // into it
                by[k] = ST::Div::scale(sums[k]);
                wide |= by[k] != 1.0f;
                sums[k] *= by[k];
            }
            rinv[k] = 1.0f / sums[k];
            rlow[k] = sums[k] > 0.0f && sums[k] <= 0x1p120f ? ST::Div::low(sums[k], rinv[k]) : 0.0f;     // (sum 0, inf, NaN: as the division)
        }
        if (std::is_same<T, bf16_t>::value && __builtin_amdgcn_ballot_w64(wide)) {
#pragma unroll
            for (int j = 0; j < V; j++)
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int w = 0; w < 4; w++) {
                        v[j][i][w] = ST::round_pair(ST::widen_bits(v[j][i][w] & 0xffffu) * by[i * R / 4], ST::widen_bits(v[j][i][w] >> 16) * by[i * R / 4]);
                        asm volatile("" : "+v"(v[j][i][w]));
                    }
            forget();
        }
        it += stride;
        const Rows done = row;
        row = rows_of(it, mrow);
#pragma unroll
        for (int j = 0; j < V; j++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                v4u q;
#pragma unroll
                for (int w = 0; w < 4; w++) q[w] = ST::short_quotients(v[j][i][w], rinv[i * R / 4], rlow[i * R / 4]);
                __builtin_amdgcn_raw_buffer_store_b128(q, ry, place(done.at[i * R / 4], j, i), 0, 2);
                v[j][i] = __builtin_amdgcn_raw_buffer_load_b128(rx, place(row.at[i * R / 4], j, i), 0, LOADS);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

// Which calls come here, against the streaming kernel (rt_softmax_stream.h); us, that one / this one, [heads, queries, keys], causal mask where one is named, inputs and
// outputs moving through 600 MB.  That one walks rows 30 (f16 rows over 4096 columns: 15) to a block, a round costs its walk whatever it holds, and the bf16 walk is
// three times the f16 one.  This one costs by the row, but reads and writes HBM less evenly than that one with its paced steps.
// What a row costs here depends on how often its sum passes a power of two: the figures are N(0, 2), N(0, 1) over 4096 columns; N(2, 3) costs
// bf16 up to a tenth more, rows sorted upwards a third ([32,1024,4096] plain 131, 132 and 176 us, there 136).
//   f16, over 4096 columns: [8,2048,8192] with a mask 134 / 126, [8,512,8192] 53 / 34, [8,700,6000] 45 / 35, [32,256,5120] 51 / 37; not where two rounds or more
//      of that kernel are nearly full ([32,480,8192] 100 / 111, [32,360,5120] with a mask 60 / 67, [32,240,8192] with a mask 65 / 70; [32,320,8192] 76 / 72).
//   f16, 2049 to 4096 columns: up to 32 rows a CU ([8,1024,3072] 30 / 26, [32,256,4096] 39 / 30; [32,224,2304] 22.4 / 23.3; [8,2048,3000] 49 / 48, [32,4096,4096] 344 / 407).
//      Against softmax16_replay_kernel, which has at most two rows to a CU: [8,64,6000] 25 / 16, [32,1,5120] 17.6 / 12.8, [32,16,4096] 17.6 / 13.8, [32,1,3000] 12.5 / 11.2, but
//      [32,1,4096] 12.6 / 12.7, [32,1,3584] 12.2 / 12.5.
//   bf16, over 4096 columns: [8,2048,8192] 201 / 124, [32,240,8192] with a mask 113 / 79.
//   bf16, 513 to 4096 columns: by what both take (sr_pays_bf16), with a mask or from 32 rows a CU or over 2048 columns, rows of whole vectors from 1025.
//   rows that are not whole vectors, up to 2048 columns: where that kernel's last round would be nearly empty ([32,1001,1001] f16 with a mask 42 / 33, bf16 60 / 46,
//      [32,1201,1201] f16 55 / 48, [16,2001,2001] f16 62 / 58; with fuller rounds f16 [32,1681,1681] 86 / 92, [32,1500,1500] 64 / 66).
inline bool sr_pays_bf16(bool mask, uint64_t period, uint64_t rows, uint32_t cols, uint64_t cus) {
    // The walk bounds the streaming kernel: 3.1 us a step and round (4.0 with a mask, 3.5 where a mask row serves two heads), and 5 us and 1.5 a step to fill and drain it;
    // a twelfth more where rows are not whole vectors.  Here 4 or 2 rows at a time on each SIMD, by the chunk of 512 or 1024 columns.  Over 650 calls of 1025 to 4096 columns the
    // pick costs half a per cent more than the better one and is never more than 3 % slower than the streaming kernel, where this one, taken for all, was slower by up to a quarter:
    // [32,1440,2560] 107 / 133, [32,480,2304] with a mask 51 / 59, [32,192,1536] with a mask 19.4 / 21.8; [32,1536,1536] with a mask 104 / 84, [32,256,4096] 60 / 41.
    const uint32_t nt = (cols + SP_TC - 1) / SP_TC, steps = nt == 7 ? 8 : nt;
    SpSched sch;
    const bool pair = sp_periods(sch, mask, period, rows, nt);
    const uint64_t rounds = sp_rounds(sch, sp_rows_per_group(sch, mask, pair, pair ? SP_HALF : SP_ROWS, cus), cus);
    double there = 5.0 + 1.5 * steps + (!mask ? 3.1 : pair ? 3.5 : 4.0) * steps * (double)rounds;
    if (cols % 8 != 0) there *= 1.08;
    const bool four = cols <= 2048;
    const uint32_t chunks = four ? nt : (cols + 1023) / 1024, at_once = four ? 16 : 8;
    const double row = four ? 0.095 + 0.085 * chunks + (mask && chunks > 2 ? 0.055 : 0.0) : 0.17 + 0.17 * chunks + (mask ? 0.06 * (chunks - 2) : 0.0);
    const double here = 11.0 + row * (double)((rows + at_once * cus - 1) / (at_once * cus) * at_once);
    return 1.04 * here < there;
}
template <typename T> bool sr_takes(bool mask, uint64_t period, uint64_t rows, uint32_t cols, uint64_t cus) {
    constexpr bool BF16 = std::is_same<T, bf16_t>::value;
    if (cols <= 512 || cols > 8192) return false;
    const bool whole = cols % 8 == 0;
    if (!whole && cols <= 2048) {
        const uint32_t steps = (cols + SP_TC - 1) / SP_TC;
        const double rounds = (double)rows / (double)(SP_ROWS * cus), full = ceil(rounds);
        if (rounds < 2.0 || full < 1.1 * rounds + 0.33 / steps || (!BF16 && full < 1.16 * rounds)) return false;
        return !BF16 || sr_pays_bf16(mask, period, rows, cols, cus);
    }
    if (BF16) {
        if (cols <= 1024 || (!whole && cols > 4096)) return false;
        if (!mask && cols <= 2048 && rows < 32 * cus) return false;
        return cols > 4096 || sr_pays_bf16(mask, period, rows, cols, cus);
    }
    if (!whole || cols <= 2048) return false;
    if (cols <= 4096) return rows <= 32 * cus && (cols <= 3072 || rows > cus / 4);
    const double rounds = (double)rows / (double)(SP_HALF * cus), full = ceil(rounds);
    if (cols > 7168 && rounds > 1.6) return full >= 1.1 * rounds && !(mask && rows <= 32 * cus);
    return rounds <= 2.5 || full >= 1.08 * rounds;
}

template <typename T, int L, int V, bool RAGGED>
int launch_row16_as(rt_device* dev, int bit, const uint16_t* table, const void* x, const void* mask, void* y, SrRows g) {
    const auto kernel = mask ? softmax16_row_kernel<T, L, V, true, RAGGED> : softmax16_row_kernel<T, L, V, false, RAGGED>;
    const uint64_t flag = 1ull << (2 * bit + (mask ? 1 : 0));
    if (!(dev->sr_attr_set & flag)) {
        if (int rc = sp_allow_lds(reinterpret_cast<const void*>(kernel))) return rc;
        dev->sr_attr_set |= flag;
    }
    // waves of a block that have rows: as many as make the rows one round, if they do
    const uint64_t cus = (uint64_t)dev->num_cus, items = ((uint64_t)g.rows * L + 63) / 64, per_cu = (items + cus - 1) / cus;
    g.waves = (uint32_t)(per_cu < (uint64_t)sr_waves(V) ? per_cu : (uint64_t)sr_waves(V));
    const uint64_t need = (items + g.waves - 1) / g.waves;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(need < cus ? need : cus)), dim3(64 * sr_waves(V)), SP_LUT_BYTES, dev->stream, table, (const T*)x, (const T*)mask,
                       (T*)y, g);
    RT_CHECK_LAUNCH("softmax16_row_kernel");
    return RT_OK;
}

template <typename T>
int launch_row16(rt_device* dev, const void* x, const void* mask, uint64_t period, void* y, uint64_t rows, uint32_t cols, bool* done) {
    *done = false;
    constexpr bool BF16 = std::is_same<T, bf16_t>::value;
    if (rows > 0x7fffffffull / (2ull * cols)) return RT_OK;              // 32-bit offsets: larger ones go in chunks there
    if (!sr_takes<T>(mask != nullptr, mask ? period : rows, rows, cols, (uint64_t)dev->num_cus)) return RT_OK;
    if (mask && rows / period % (cols > 2048 ? 2 : 4) != 0) return RT_OK;        // the rows of a wave share a mask row
    if (dev->debug_softmax_pace) return RT_OK;                           // a pace set by hand is the streaming kernel's
    // the exp table is built on first use, which synchronises: not while a graph is being captured
    if (dev->capturing && !dev->unary_lut[BF16][RT_EXP]) return RT_OK;
    const uint16_t* table = nullptr;
    if (int rc = rt_unary_table(dev, BF16, RT_EXP, &table)) return rc;
    SrRows g;
    g.rows = (uint32_t)rows;
    g.cols = cols;
    g.period = (uint32_t)(mask ? period : rows);
    g.reps_div = make_fastdiv((uint32_t)(mask ? rows / period : 1));
    const int chunks = (int)(cols > 2048 ? (cols + 1023) / 1024 : (cols + 511) / 512);
    int rc = RT_OK;
#define RT_SR(LC, VC, RG, BIT)                                                                                     \
    case VC:                                                                                                       \
        rc = launch_row16_as<T, LC, VC, RG>(dev, (BIT) + (BF16 ? 9 : 0), table, x, mask, y, g);                    \
        break
#define RT_SR_NONE default: return rt_fail(RT_ERR_ARG, "softmax: internal: %u columns for several rows to a wave", cols)
    if (cols % 8 != 0 && cols <= 2048) {
        switch (chunks) { RT_SR(16, 2, true, 0); RT_SR(16, 3, true, 1); RT_SR(16, 4, true, 2); RT_SR_NONE; }
    } else if (cols > 2048 && cols % 8 == 0) {
        switch (chunks) {
            RT_SR(32, 3, false, 3); RT_SR(32, 4, false, 4); RT_SR(32, 5, false, 5); RT_SR(32, 6, false, 6); RT_SR(32, 7, false, 7); RT_SR(32, 8, false, 8);
            RT_SR_NONE;
        }
    } else if constexpr (BF16) {
        if (cols > 2048) {
            switch (chunks) { RT_SR(32, 3, true, 9); RT_SR(32, 4, true, 10); RT_SR_NONE; }
        } else {
            switch (chunks) { RT_SR(16, 3, false, 11); RT_SR(16, 4, false, 12); RT_SR_NONE; }
        }
    }
#undef RT_SR_NONE
#undef RT_SR
    *done = rc == RT_OK;
    return rc;
}

}  // namespace

int rt_softmax_row(rt_device* dev, bool bf16, const void* x, const void* mask, uint64_t period, void* y, uint64_t rows, uint32_t cols, bool* done) {
    return bf16 ? launch_row16<bf16_t>(dev, x, mask, period, y, rows, cols, done) : launch_row16<half_t>(dev, x, mask, period, y, rows, cols, done);
}
