// The tolerance-mode solve in one launch: the state machine of cg.hip
// (k_cg_spmv and k_cg_update, whose arithmetic and rounding it repeats
// operation by operation), with a cloth's rows kept by the workgroups that
// own them for the whole solve.
//
// What bounds it.  A cloth solved by two launches an iteration waits on the
// launches: 9.1 us an iteration for a 125 x 125 cloth whose 6 MB of matrix
// would stream in 1 us, 15.0 us for 257 x 257.  Here one workgroup keeps up
// to 8 slices (512 rows; 4 in FP64): its matrix blocks stay in registers (13
// slots of 9 values a lane), its directions and those of the rows around it
// in LDS, and r, z, q, P and the solution's increments in registers, so that
// an iteration reads no matrix and waits only for the two sums (d.q; r.z and
// r.r) that every part of the cloth needs, and for its neighbours' z.  Per
// iteration: 21 x 21 (one part) 9.0 -> 3.3 us, 125 x 125 (31 parts) 9.1 ->
// 5.4, 257 x 257 (130) 15.0 -> 9.3, 190 x 211 in FP64 (157) 16.0 -> 9.3.  Of
// the 125 x 125 cloth's, 2.7 us are the two exchanges (a value is visible to
// another workgroup some 0.8 us after its store), the rest chains of
// dependent instructions: the product 0.5, the sums 1.1, the update and the
// directions 0.5, two FP64 divisions 0.2.
//
// Exchange between workgroups.  Every exchanged 32-bit half of a value
// travels in one 64-bit word with a tag, the number of the exchange, written
// and read by relaxed agent-scope atomics: a reader polls the word itself
// until it carries the tag it expects, so a value needs no flag, fence or
// cache write-back beside it (agent-scope fences write back and invalidate
// L2 and cost 23 us a phase when a persistent form was tried with them).  A
// word is written again only after every reader is known to have read it:
// between two writes of a word by the same workgroup lies an exchange of sums
// in which each workgroup of the cloth publishes after its own reads (for
// the words of a true residual, whose solution values are exchanged between
// neighbours only, the column structure's symmetry gives the same: who reads
// a part's rows is read by it).  Tags continue from solve to solve
// (ResidentBatch::epoch).
//
// Workgroups take tickets in order (ResidentCtl::next), one part each, a
// cloth's parts in a row.  A workgroup that holds a ticket is running, so
// whenever the grid's first `parts` workgroups of a cloth fit on the chip
// together (resident_capacity; the host checks it) the earliest unfinished
// cloth has all of its parts running, and the launch ends.  Other work on
// the device may delay a workgroup, so every wait is bounded all the same
// (ResidentCtl::wait_ticks, counted while no cloth of the launch gets on: a
// later cloth's parts may wait through whole solves of earlier ones); a wait
// that runs out sets ResidentCtl::aborted, every workgroup leaves, and the host
// solves again by launches.
//
// The reference's semantics (solver_mode "reference": FP64, exactly
// max_iters - 1 iterations, BaraffCloth.cpp:529) are the same recurrences
// with a tolerance of 0 and that cap, and the true residual after the last
// iteration is the one that the counters report; REF gives it pcg.hip's
// rounding, bit for bit.  65 x 65, 199 iterations, assembly included: 13.8
// us an iteration by pcg.hip's launches, 6.4 here.
//
// PAUSE, for the server's rounds: after a number of iterations a solve leaves
// the launch (the recurrences' vectors and scalars to memory), so that a short
// request need not wait for a long one's solve, and the next launch goes on as
// if nothing had been between.
//
// Same rounding as cg.hip: a row's slots are added per lane phase of the
// variant with L lanes per row, then the phases; a slice's partial sums in
// that variant's order (slice_sum); a cloth's sums over its slices as
// wave_sets_sum adds them.  Results are therefore bit-identical to those of
// the launches, alone and in any batch.
#include <algorithm>

#include "cg_math.h"
#include "reduce.h"
#include "resident.h"

namespace bw
{
namespace
{

typedef unsigned long long u64;

__device__ inline u64 word_load(const G<u64> *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void word_store(G<u64> *p, unsigned tag, unsigned value)
{
    __hip_atomic_store(p, (u64)tag << 32 | value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned word_tag(u64 w) { return (unsigned)(w >> 32); }

// 32-bit pieces of a value, and back
template <typename T> struct Pieces;
template <> struct Pieces<float>
{
    static constexpr int N = 1;
    __device__ static unsigned get(float v, int) { return __float_as_uint(v); }
    __device__ static float join(const u64 *w) { return __uint_as_float((unsigned)w[0]); }
};
template <> struct Pieces<double>
{
    static constexpr int N = 2;
    __device__ static unsigned get(double v, int k)
    {
        return k ? (unsigned)__double2hiint(v) : (unsigned)__double2loint(v);
    }
    __device__ static double join(const u64 *w)
    {
        return __hiloint2double((int)(unsigned)w[1], (int)(unsigned)w[0]);
    }
};

__device__ inline int control(const int *p)
{
    return __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// A bounded wait: true once the time given has passed without progress
// anywhere in the launch (a part may wait for a whole solve of the cloths
// before its own, whose end gives the other parts of its cloth their CUs), or
// another workgroup has given up (looked at every 64 polls)
struct Patience
{
    const ResidentCtl *ctl;
    u64 since;
    int polls, seen;
    __device__ bool out()
    {
        if (++polls & 63)
            return false;
        const u64 t = wall_clock64();
        const int now = control(&ctl->next) + control(&ctl->progress);
        if (!since || now != seen)
        {
            since = t;
            seen = now;
        }
        return t - since > ctl->wait_ticks || control(&ctl->aborted) != 0;
    }
};
// Iterations of an FP64 cloth after which ResidentCtl::progress moves.  A
// mixed one's moves with every eighth true residual, 33,000 iterations or 0.6 s
// at most (with every one 5 x 5 and 21 x 21 lost 1.5%, with a test in each
// iteration 2%).
constexpr int PROGRESS = 256;

// v, but unknown to the compiler: addresses formed from it are formed where
// they are used instead of being kept in registers across the solve
__device__ inline int here(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// word i of words, by a scalar base and a 32-bit offset
__device__ inline G<u64> *word_at(G<u64> *words, unsigned i)
{
    return reinterpret_cast<G<u64> *>(reinterpret_cast<G<char> *>(words) + 8u * i);
}

// Waits until the K words that `at` gives (at(k): a word's address) carry the
// tag, in every lane of the wavefront
template <int K, typename At>
__device__ inline bool await(u64 (&v)[K], unsigned tag, Patience w, const At &at)
{
    for (;;)
    {
        bool all = true;
#pragma unroll
        for (int k = 0; k < K; k++)
            v[k] = word_load(at(k));
#pragma unroll
        for (int k = 0; k < K; k++)
            all = all & (word_tag(v[k]) == tag);
        if (__all(all))
            return true;
        if (w.out())
            return false;
    }
}

// All n words p[0 .. n-1] by the workgroup's NT threads, their values to dst
// (LDS), K in flight a lane; lanes past the end poll the last word.  With
// the last of them, waits for the H words x at x_at(h) that carry x_tag:
// their publishers store them before the words of p, so they are there in
// the same round trip.
template <int K, int NT, int H, typename At>
__device__ inline bool pull_words(G<u64> *p, int n, unsigned tag, unsigned *dst, Patience w,
                                  u64 (&x)[H], unsigned x_tag, const At &x_at, bool x_any)
{
#pragma clang loop unroll(disable)
    for (int i = here(threadIdx.x);; i += K * NT)
    {
        if ((i & ~63) >= n && !x_any)
            return true;
        // (waves past the end have only x to wait for)
        const bool some = (i & ~63) < n;
        const bool last = (i & ~63) + K * NT >= n && x_any;
        u64 v[K];
#pragma unroll
        for (int k = 0; k < K; k++)
            v[k] = some ? word_load(word_at(p, min(i + k * NT, n - 1))) : (u64)tag << 32;
        if (last)
#pragma unroll
            for (int h = 0; h < H; h++)
                x[h] = word_load(x_at(h));
        for (;;)
        {
            bool all = true;
#pragma unroll
            for (int k = 0; k < K; k++)
                all = all & (word_tag(v[k]) == tag);
            if (last)
#pragma unroll
                for (int h = 0; h < H; h++)
                    all = all & (word_tag(x[h]) == x_tag);
            if (__all(all))
                break;
            if (w.out())
                return false;
#pragma unroll
            for (int k = 0; k < K; k++)
                if (word_tag(v[k]) != tag)
                    v[k] = word_load(word_at(p, min(i + k * NT, n - 1)));
            if (last)
#pragma unroll
                for (int h = 0; h < H; h++)
                    if (word_tag(x[h]) != x_tag)
                        x[h] = word_load(x_at(h));
        }
#pragma unroll
        for (int k = 0; k < K; k++)
            if (i + k * NT < n)
                dst[i + k * NT] = (unsigned)v[k];
        if ((i & ~63) + K * NT >= n)
            return true;
    }
}

// a value that every lane holds, as a scalar (kept in scalar registers
// across the solve: the matrix fills the vector registers)
__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline double uniform(double v)
{
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// v of lane l (uniform)
__device__ inline double lane_value(double v, int l)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// A slice's sum over its 64 rows, lane l holding row l, in the order of the
// launches' variant with L lanes per row: that variant sums 64 / L rows in
// each of L wavefronts, then the wavefronts in order.
template <int L> __device__ inline double slice_sum(double v)
{
    if constexpr (L == 1)
        return wave_sum(v);
    if constexpr (L == 2)
        v = swap_add<16>(v, v);
    v = row_sum(v);
    if constexpr (L == 2)
        return lane_value(v, 0) + lane_value(v, 32);
    return ((lane_value(v, 0) + lane_value(v, 16)) + lane_value(v, 32)) + lane_value(v, 48);
}

// The order of pcg.hip's reduce_cloth over the n sets of N sums in LDS (one a
// solver workgroup there): a wavefront's worth of sets at a time, four of
// those in turn.
template <int N> __device__ inline void block_sets_sum(const double *sm, int n, double (&out)[N])
{
    const int lane = threadIdx.x & 63;
    for (int j = 0; j < N; j++)
        out[j] = 0.0;
#pragma clang loop unroll(disable)
    for (int g = 0; g < 4 && 64 * g < n; g++)
        for (int j = 0; j < N; j++)
        {
            double t = 0.0;
            for (int s = 64 * g + lane; s < n; s += 256)
                t += sm[N * s + j];
            out[j] += uniform(wave_sum(t));
        }
}

// wave_sets_sum over the n sets of N sums in LDS, as scalars.  Four sets a
// lane at a time; past the end zeros, which change no sum.
template <int N> __device__ inline void sets_sum(const double *sm, int n, double (&out)[N])
{
    const int lane = threadIdx.x & 63;
    double t[N];
    for (int j = 0; j < N; j++)
        t[j] = 0.0;
#pragma clang loop unroll(disable)
    for (int s0 = lane; (s0 & ~63) < n; s0 += 256)
    {
        double a[4][N];
#pragma unroll
        for (int u = 0; u < 4; u++)
            for (int j = 0; j < N; j++)
                a[u][j] = sm[N * min(s0 + 64 * u, n - 1) + j];
#pragma unroll
        for (int u = 0; u < 4; u++)
            for (int j = 0; j < N; j++)
                t[j] += s0 + 64 * u < n ? a[u][j] : 0.0;
    }
    if constexpr (N == 1)
        out[0] = uniform(wave_sum(t[0]));
    else
    {
        const double v = wave_sum2(t[0], t[1]);
        out[0] = lane_value(v, 0);
        out[1] = lane_value(v, 32);
        if constexpr (N == 3)
            out[2] = uniform(wave_sum(t[2]));
    }
}

// the row's phases of the variant with L lanes per row
template <int L, typename T> __device__ inline T phases(const T (&y)[L])
{
    if constexpr (L == 1)
        return y[0];
    else if constexpr (L == 2)
        return y[0] + y[1];
    else
        return (y[0] + y[1]) + (y[2] + y[3]);
}

// block_row, or the order in which pcg.hip's compiler fuses its sum of three
// products: m2 v2 + (m0 v0 + (m1 v1))
template <bool REF, typename T> __device__ inline T block(T m0, T m1, T m2, T v0, T v1, T v2)
{
    return REF ? fma_t(m2, v2, fma_t(m0, v0, m1 * v1)) : block_row<T>(m0, m1, m2, v0, v1, v2);
}

__device__ inline ResidentPart uniform_part(const ResidentPart &v)
{
    ResidentPart p;
    p.inst = uniform(v.inst);
    p.slice0 = uniform(v.slice0);
    p.n_slices = uniform(v.n_slices);
    p.sets = uniform(v.sets);
    p.set0 = uniform(v.set0);
    p.halo_off = uniform(v.halo_off);
    p.halo_n = uniform(v.halo_n);
    p.parts = uniform(v.parts);
    return p;
}

// WAVES wavefronts, a slice each.  The matrix takes 117 vector registers of
// 256 in the mixed form with two wavefronts a SIMD (234 of 512 in FP64 with
// one), so the rest is kept small: what only a true residual needs stays in
// LDS or memory, what is uniform in scalar registers, and addresses are
// formed where they are used (here()); with spills to scratch the product
// alone took 5,500 cycles an iteration instead of 1,150.  The compiler keeps
// 65 to 88 scalars in lanes of a vector register all the same (moved back one
// by one, most of them in the exchange and at a true residual), and in FP64
// 154 to 166 of the matrix's registers in the accumulator file, copied back
// before each product; no variant with 1 or 2 lanes per row spills vectors.
// REF: the reference's semantics with pcg.hip's rounding (T = double, L = 1):
// its order of a block's three products, and one set of sums per workgroup.
template <typename T, int WAVES, int L, bool REF, bool PAUSE = false>
__global__ void __launch_bounds__(WAVES * 64)
k_resident(ResidentLaunch a)
{
    static_assert(!REF || (WAVES == BW_SB && L == 1), "a part is one of pcg.hip's workgroups");
    constexpr int NT = WAVES * 64; // threads, and rows of a part
    constexpr int NP = Pieces<T>::N;
    constexpr bool MIXED = sizeof(T) == sizeof(float);
    extern __shared__ __align__(16) unsigned char rs_lds[];
    __shared__ int sh_ticket, sh_failed;
    __shared__ int sh_stop; // PAUSE: iterations of the solve at which it pauses
    __shared__ CgState sh_st;
    // REF: the slices' sums of this part, apart from the parts' sums, which
    // the other wavefronts gather while the first one adds these
    __shared__ double sh_slices[REF ? 3 * WAVES : 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
    const int E = NT + a.halo_max;
    T *dl = reinterpret_cast<T *>(rs_lds);               // directions, 3 an entry
    double *xl = reinterpret_cast<double *>(dl + 3 * E); // solution, 3 an entry
    double *sm_dq = xl + 3 * E;                          // a set's sums: 1 value
    double *sm_rz = sm_dq + a.sets_max;                  // 2 values (3 after a true residual)
    int *hrow = reinterpret_cast<int *>(sm_rz + 3 * a.sets_max); // the halo's rows
    // blocks of slots past the registers' (planes as in W), a.extra of a
    // slice, and their offsets into dl
    T *mx = reinterpret_cast<T *>(hrow + a.halo_max);
    unsigned *cx = reinterpret_cast<unsigned *>(mx + a.extra * 9 * SLICE);
    const int2 *ticket = reinterpret_cast<const int2 *>(a.ctl + 1);
    const Patience patience = {a.ctl, 0, 0, 0};
    // every wavefront here, and no wait of the workgroup has run out
    auto meet = [&]() {
        __syncthreads();
        return sh_failed == 0;
    };

    for (;;)
    {
        __syncthreads();
        if (tid == 0)
        {
            sh_ticket = atomicAdd(&a.ctl->next, 1);
            sh_failed = 0;
        }
        __syncthreads();
        if (sh_ticket >= a.tickets)
            return;
        const int2 tk = ticket[uniform(sh_ticket)];
        const ResidentBatch &rb = a.table[uniform(tk.x)];
        const DeviceBatch &d = rb.d;
        const ResidentPart pt = uniform_part(rb.part[uniform(tk.y)]);
        const int inst = pt.inst;
        // The cloth's state as k_cg_spmv and k_cg_update keep it, brought up
        // to date at each true residual, in LDS; in between, an iteration
        // needs these scalars only.
        if (tid == 0)
            sh_st = load_state(glob(d.cg) + 2 * inst);
        __syncthreads();
        if (sh_st.done)
            continue;
        int steps = 0;       // iterations since the last true residual
        int room = 0;        // after which the next is due
        double enough = 0.0; // r.r at which it is due
        double rho = 0.0;    // r.(P r) of the current direction
        bool first = true;   // the next direction is P r
        bool w64 = uniform(sh_st.w64) != 0;
        bool check = true;   // a true residual is due (the warm start's)
        bool due = true;     // PAUSE: whatever the counts
        // sets of sums: one a slice, or one a part
        const int sets = REF ? pt.parts : pt.sets;
        const int set_base = REF ? pt.set0 / BW_SB : pt.set0;
        const bool shared = pt.parts > 1;
        const bool have = wave < pt.n_slices; // this wavefront has a slice
        const int sl = pt.slice0 + (have ? wave : 0);
        const int ws = have ? uniform(d.slice_w[sl]) : 0; // its width
        const int base = uniform(d.slice_off[sl]);        // its first ELL entry
        auto row = [&]() { return (unsigned)here(sl * SLICE + lane); };
        unsigned tag = (unsigned)uniform((int)rb.epoch[inst]);

        // the rows' matrix blocks and column positions; slots past the
        // slice's width: zero blocks on the row itself
        T m[RS_SLOTS][9];
        unsigned c[(RS_SLOTS + 1) / 2]; // byte offsets into dl, two a register
        T P[3], r[3], z[3], dv[3];
        float x32[3] = {0.0f, 0.0f, 0.0f};
        double x64[3]; // FP64 form (the mixed form's stays in memory)
        {
            const G<uint16_t> *pos = glob(rb.pos) + base;
            const G<T> *W = glob(Vecs<T>::W(d)) + 9 * (size_t)base;
#pragma unroll
            for (int k = 0; k < RS_SLOTS; k++)
            {
                unsigned at = tid;
                if (k < ws)
                    at = pos[k * SLICE + lane];
                at *= 3 * sizeof(T);
                c[k / 2] = k & 1 ? c[k / 2] | at << 16 : at;
                for (int q = 0; q < 9; q++)
                    m[k][q] = k < ws ? W[(9 * k + q) * SLICE + lane] : (T)0;
            }
        }
        // the slots past them go to LDS while it lasts, the part's slices in
        // order: this slice's are x0 .. x0 + nx - 1 (as many for each slice as
        // the widest has: LDS holds too few, Delaunay clothes of 14,430 points
        // 8.3 us an iteration against 6.9, of 60,000 10.7 against 9.6, of
        // 6,000 in FP64 8.5 against 7.8)
        int x0 = 0;
        for (int i = 0; i < wave; i++)
            x0 += max(0, (i < pt.n_slices ? uniform(d.slice_w[pt.slice0 + i]) : 0) - RS_SLOTS);
        const int nx = max(0, min(ws - RS_SLOTS, a.extra - x0));
        {
            const G<uint16_t> *pos = glob(rb.pos) + base + RS_SLOTS * SLICE + lane;
            const G<T> *W = glob(Vecs<T>::W(d)) + 9 * ((size_t)base + RS_SLOTS * SLICE) + lane;
#pragma clang loop unroll(disable)
            for (int k = 0; k < nx; k++)
            {
                cx[(x0 + k) * SLICE + lane] = 3 * (unsigned)sizeof(T) * pos[k * SLICE];
                for (int q = 0; q < 9; q++)
                    mx[(9 * (x0 + k) + q) * SLICE + lane] = W[(9 * k + q) * SLICE];
            }
        }
        for (int i = 0; i < 3; i++)
        {
            P[i] = have ? glob(Vecs<T>::P(d))[3 * row() + i] : (T)0;
            x64[i] = !MIXED && have ? glob(d.dx)[3 * row() + i] : 0.0;
            r[i] = z[i] = dv[i] = (T)0;
        }
        for (int i = tid; i < pt.halo_n; i += NT)
            hrow[i] = rb.halo_row[pt.halo_off + i];
        __syncthreads();

        // exchange words; those of rows are planes, one per component and
        // piece
        G<u64> *const words_z = glob(rb.z), *const words_dq = glob(rb.s_dq),
                *const words_rz = glob(rb.s_rz);
        const unsigned plane = (unsigned)d.n_rows;
        double rz = 0.0, rr = 0.0; // the last exchange's sums
        unsigned z_tag = 0;        // the exchange that carried z
        u64 hz[3 * NP];            // z of the halo entry that this thread takes first

        // z of this part's rows to the others
        auto publish_z = [&]() {
            z_tag = tag;
            if (!shared || !have)
                return;
            const unsigned p = row();
            for (int i = 0; i < 3; i++)
                for (int h = 0; h < NP; h++)
                    word_store(word_at(words_z, (i * NP + h) * plane + p), tag,
                               Pieces<T>::get(z[i], h));
        };
        // word w (piece w % pieces of component w / pieces) of halo entry e
        auto halo_word = [&](G<u64> *words, int e, int w) {
            return word_at(words, w * plane + (unsigned)hrow[min(e, pt.halo_n - 1)]);
        };
        // The wavefront's sums of its slice, 64 / span of them: lane l holds
        // number l / span, in all span lanes.  The part's sums meet in LDS and
        // go out as one store, so that a line of words has one writer and
        // one write (257 x 257: 9.3 us an iteration against 10.2 with a
        // store per wavefront; smaller cloths within 4%).
        auto publish = [&](double v, int span, int n, G<u64> *words, double *sm) {
            const int l = here(lane), at = l / span;
            if constexpr (REF)
            {
                // pcg.hip's block_sum: the wavefronts in order
                if (have && at < n && l % span == 0)
                    sh_slices[n * wave + at] = v;
                __syncthreads();
                const int t = here(tid);
                if (t >= 2 * n || (!shared && (t & 1)))
                    return;
                const double *from = sh_slices + t / 2;
                const double sum = ((from[0] + from[n]) + from[2 * n]) + from[3 * n];
                if (!shared)
                    sm[t / 2] = sum;
                else
                    word_store(word_at(words, 2 * n * (pt.slice0 / BW_SB) + t), tag,
                               (unsigned)(t & 1 ? __double2hiint(sum) : __double2loint(sum)));
                return;
            }
            if (have && at < n && l % span == 0)
                sm[n * (sl - pt.set0) + at] = v;
            if (!shared)
                return;
            __syncthreads();
            const int t = here(tid);
            const unsigned *from =
                reinterpret_cast<const unsigned *>(sm + n * (pt.slice0 - pt.set0));
            if (t < 2 * n * pt.n_slices)
                word_store(word_at(words, 2 * n * pt.slice0 + t), tag, from[t]);
        };
        // every slice's n sums to LDS; with_z: and the first entries of the
        // halo's z to hz
        auto gather = [&](int n, G<u64> *words, double *sm, bool with_z) {
            if (!shared)
                return;
            unsigned *dst = reinterpret_cast<unsigned *>(sm);
            G<u64> *w = words + (size_t)set_base * n * 2;
            const int count = sets * n * 2;
            with_z = with_z && pt.halo_n > 0;
            const int e = here(tid);
            auto at = [&](int h) { return halo_word(words_z, e, h); };
            bool in_time;
            if (count <= NT)
                in_time = pull_words<1, NT>(w, count, tag, dst, patience, hz, z_tag, at, with_z);
            else if (count <= 2 * NT)
                in_time = pull_words<2, NT>(w, count, tag, dst, patience, hz, z_tag, at, with_z);
            else
                in_time = pull_words<5, NT>(w, count, tag, dst, patience, hz, z_tag, at, with_z);
            if (!in_time)
                sh_failed = 1;
        };
        auto total = [&](const double *sm, auto &out) {
            constexpr int N = sizeof(out) / sizeof(out[0]);
            if constexpr (REF)
                block_sets_sum<N>(sm, sets, out);
            else
                sets_sum<N>(sm, sets, out);
        };
        // the slice's rows of W64 times the vectors v of the LDS array, in
        // the order of the variant with L lanes per row
        // slots whose blocks are read together: 3 with one lane per row (4
        // spill), else one by one.  The FP64 matrix comes from memory, a trip
        // a round: with all iterations on it 257 x 257 26.3 -> 18.5 us an
        // iteration, 125 x 125 12.4 -> 12.1 (10.3 by launches: there a CU
        // streams 470 KB an iteration), 21 x 21 9.3 -> 8.3; a 5 x 5 cloth's
        // step, 7 true residuals, 333 -> 305 us
        constexpr int C64 = L == 1 ? 3 : 1;
        auto product64 = [&](const auto *v, double (&sum)[3]) {
            double y[3][L] = {};
            const G<uint16_t> *pos = glob(rb.pos) + base + here(lane);
            const G<double> *W64 = glob(d.W64) + 9 * (size_t)base + here(lane);
#pragma clang loop unroll(disable)
            for (int k0 = 0; k0 < ws; k0 += C64 * L)
            {
                if constexpr (C64 == 1)
                {
#pragma unroll
                    for (int j = 0; j < L; j++)
                        if (k0 + j < ws)
                        {
                            const auto *x = v + 3 * (int)pos[(k0 + j) * SLICE];
                            const G<double> *w = W64 + 9 * (k0 + j) * SLICE;
                            for (int i = 0; i < 3; i++)
                                y[i][j] += block<REF>(w[(3 * i) * SLICE], w[(3 * i + 1) * SLICE],
                                                      w[(3 * i + 2) * SLICE], (double)x[0],
                                                      (double)x[1], (double)x[2]);
                        }
                }
                else
                {
                    double w[C64][9];
                    int at[C64];
#pragma unroll
                    for (int c = 0; c < C64; c++)
                    {
                        const int k = min(k0 + c, ws - 1);
                        at[c] = 3 * (int)pos[k * SLICE];
                        for (int q = 0; q < 9; q++)
                            w[c][q] = W64[(9 * k + q) * SLICE];
                    }
#pragma unroll
                    for (int c = 0; c < C64; c++)
                        if (k0 + c < ws)
                            for (int i = 0; i < 3; i++)
                                y[i][0] += block<REF>(w[c][3 * i], w[c][3 * i + 1],
                                                      w[c][3 * i + 2], (double)v[at[c]],
                                                      (double)v[at[c] + 1], (double)v[at[c] + 2]);
                }
            }
            for (int i = 0; i < 3; i++)
                sum[i] = phases<L>(y[i]);
        };

        if constexpr (PAUSE)
        {
            const CgState &st = sh_st;
            if (tid == 0)
                sh_stop = st.total + (st.start ? 0 : st.since) + a.pause;
            __syncthreads();
            if (uniform(st.start) == 0)
            {
                // on from where an earlier launch left the solve (below); the
                // state holds r.z in rr_true's place
                check = due = first = false;
                steps = uniform(st.since);
                rho = uniform(st.rho);
                rz = uniform(st.rr_true);
                rr = uniform(st.rr);
                const G<InstParams> *ip = glob(d.params) + inst;
                room = uniform(min(min(ip->max_iter - st.total, ip->max_since),
                                   sh_stop - st.total));
                enough = uniform(fmax(ip->tol * ip->tol * st.bb, ip->rel2 * st.rr_ref));
                const G<T> *dp = glob(Vecs<T>::d0(d));
                for (int i = 0; i < 3; i++)
                {
                    r[i] = have ? glob(Vecs<T>::r(d))[3 * row() + i] : (T)0;
                    dv[i] = have ? dp[3 * row() + i] : (T)0;
                    if constexpr (MIXED)
                        x32[i] = have ? glob(d.dx32)[3 * row() + i] : 0.0f;
                    z[i] = P[i] * r[i];
                }
                for (int e = tid; e < pt.halo_n; e += NT)
                    for (int i = 0; i < 3; i++)
                        dl[3 * (NT + e) + i] = dp[3 * hrow[e] + i];
                ++tag;
                publish_z();
                // (the other halo entries' z are awaited where they are used)
                const int e = here(tid);
                if ((e & ~63) < pt.halo_n &&
                    !await<3 * NP>(hz, z_tag, patience,
                                   [&](int w) { return halo_word(words_z, e, w); }))
                    sh_failed = 1;
            }
        }

        bool failed = false, paused = false;
        for (;;)
        {
            if (check)
            {
                if constexpr (PAUSE)
                {
                    const G<InstParams> *ip = glob(d.params) + inst;
                    paused = !due && rr > enough && rr < __builtin_inf() &&
                             steps < uniform(min(ip->max_iter - sh_st.total, ip->max_since));
                    if (paused)
                        break;
                    due = false;
                }
                // r = b - W64 (dx + dx32), z = P r: the solution of the
                // part's own rows and of its halo through LDS
                ++tag;
                for (int i = 0; i < 3; i++)
                {
                    double x = x64[i];
                    if (MIXED && have)
                    {
                        // (the mixed form's FP64 solution changes here only,
                        // and stays in memory in between)
                        G<double> *x_own = glob(d.dx) + 3 * row() + i;
                        x = *x_own + (double)x32[i];
                        *x_own = x;
                        x32[i] = 0.0f;
                    }
                    xl[3 * tid + i] = x;
                    if (shared && have)
                        for (int h = 0; h < 2; h++)
                            word_store(word_at(glob(rb.x), (2 * i + h) * plane + row()), tag,
                                       Pieces<double>::get(x, h));
                }
                bool in_time = true;
#pragma clang loop unroll(disable)
                for (int e = here(tid); (e & ~63) < pt.halo_n && in_time; e += NT)
                {
                    u64 x[6];
                    in_time = await<6>(x, tag, patience,
                                       [&](int w) { return halo_word(glob(rb.x), e, w); });
                    if (e < pt.halo_n)
                        for (int i = 0; i < 3; i++)
                            xl[3 * (NT + e) + i] = Pieces<double>::join(x + 2 * i);
                }
                if (!in_time)
                    sh_failed = 1;
                if (!meet())
                {
                    failed = true;
                    break;
                }
                ++tag;
                double y[3], v[3] = {0.0, 0.0, 0.0};
                product64(xl, y);
                for (int i = 0; i < 3; i++)
                {
                    const double bv = have ? glob(d.b)[3 * row() + i] : 0.0;
                    const double rv = bv - y[i];
                    r[i] = (T)rv;
                    z[i] = P[i] * r[i];
                    v[0] = fma_t((double)r[i], (double)z[i], v[0]);
                    v[1] = fma_t(rv, rv, v[1]);
                    v[2] = fma_t(bv, bv, v[2]);
                }
                publish_z();
                {
                    const double s0 = slice_sum<L>(v[0]), s1 = slice_sum<L>(v[1]),
                                 s2 = slice_sum<L>(v[2]);
                    publish(lane < 16 ? s0 : lane < 32 ? s1 : s2, 16, 3, glob(rb.s_res), sm_rz);
                }
                gather(3, glob(rb.s_res), sm_rz, true);
                if (!meet())
                {
                    failed = true;
                    break;
                }
                double t[3];
                total(sm_rz, t);
                rz = t[0];
                rr = t[1];
                // stop, or go on from the true residual (k_cg_spmv after a
                // pending one)
                CgState st = sh_st;
                const G<InstParams> *ip = glob(d.params) + inst;
                const double tol2 = ip->tol * ip->tol;
                st.total += steps;
                st.since = steps;
                st.updates += 1;
                st.start = 0;
                st.bb = t[2];
                st.rr_true = rr;
                st.done = rr <= tol2 * st.bb || st.final_check || st.total >= ip->max_iter ||
                          !isfinite(rr);
                if (!st.done && ip->stall > 0.0 && !w64 && st.since >= ip->max_since &&
                    rr > ip->stall * st.rr_ref)
                    w64 = first = true;
                st.rr_ref = rr;
                st.w64 = w64;
                __syncthreads();
                if (tid == 0)
                {
                    sh_st = st;
                    if (pt.slice0 == pt.set0 && (st.updates & 7) == 0)
                        atomicAdd(&a.ctl->progress, 1);
                }
                if (uniform(st.done))
                    break;
                steps = 0;
                room = uniform(min(ip->max_iter - st.total, ip->max_since));
                if constexpr (PAUSE)
                    room = min(room, uniform(sh_stop - st.total));
                enough = uniform(fmax(tol2 * st.bb, ip->rel2 * rr));
                check = false;
                bool leave;
                if constexpr (MIXED) // (one scalar: 21 x 21 4% faster than branches)
                    leave = uniform(a.give_up > 0
                                        ? st.total >= a.give_up
                                        : a.give_up < 0 && st.w64 && st.since > 0 && first);
                else
                    leave = a.give_up > 0 && st.total >= a.give_up;
                if (leave)
                {
                    failed = true;
                    break;
                }
            }
            const double beta = first ? 0.0 : uniform(rz / rho);
            if (REF && !first && beta == 0.0)
            {
                // the reference stops here (BaraffCloth.cpp:585-590)
                if (tid == 0)
                    sh_st.final_check = 1;
                check = true;
                continue;
            }
            rho = rz;

            // d = z + beta d_prev of the part's rows and of its halo
            const T bt = (T)beta;
            for (int i = 0; i < 3; i++)
            {
                dv[i] = dir_value<T>(z[i], dv[i], bt, first);
                dl[3 * tid + i] = dv[i];
            }
            bool in_time = true;
#pragma clang loop unroll(disable)
            for (int e = here(tid), n = 0; (e & ~63) < pt.halo_n && in_time; e += NT, n++)
            {
                // (the first entries' z came with the sums)
                if (n > 0)
                    in_time = await<3 * NP>(hz, z_tag, patience,
                                            [&](int w) { return halo_word(words_z, e, w); });
                if (e < pt.halo_n)
                {
                    T *p = dl + 3 * (NT + e);
                    for (int i = 0; i < 3; i++)
                        p[i] = dir_value<T>(Pieces<T>::join(hz + i * NP), p[i], bt, first);
                }
            }
            if (!in_time)
                sh_failed = 1;
            if (!meet())
            {
                failed = true;
                break;
            }
            // q = W d
            T q[3];
            ++tag;
            if (MIXED && w64)
            {
                // the FP64 matrix under FP32 vectors, from memory
                double y[3];
                product64(dl, y);
                for (int i = 0; i < 3; i++)
                    q[i] = (T)y[i];
            }
            else
            {
                T y[3][L] = {};
                auto slots = [&](auto first_slot, auto count) {
                    constexpr int K0 = decltype(first_slot)::value, N = decltype(count)::value;
                    T x[N][3];
#pragma unroll
                    for (int k = 0; k < N; k++)
                    {
                        const unsigned at =
                            (K0 + k) & 1 ? c[(K0 + k) / 2] >> 16 : c[(K0 + k) / 2] & 0xffff;
                        const T *p = reinterpret_cast<const T *>(rs_lds + at);
                        for (int i = 0; i < 3; i++)
                            x[k][i] = p[i];
                    }
#pragma unroll
                    for (int k = 0; k < N; k++)
                        for (int i = 0; i < 3; i++)
                            y[i][(K0 + k) % L] +=
                                block<REF>(m[K0 + k][3 * i], m[K0 + k][3 * i + 1],
                                           m[K0 + k][3 * i + 2], x[k][0], x[k][1], x[k][2]);
                };
                slots(std::integral_constant<int, 0>(), std::integral_constant<int, 9>());
                if (ws > 9)
                    slots(std::integral_constant<int, 9>(),
                          std::integral_constant<int, RS_SLOTS - 9>());
                // rows wider than the registers hold: the blocks in LDS, then
                // the rest from memory (a 20,011-point mesh with rows of up
                // to 21 blocks: 7.0 us an iteration, 8.5 with all of them
                // from memory)
                auto add = [&](int k, T (&t)[3]) __attribute__((always_inline)) {
#pragma unroll
                    for (int j = 0; j < L; j++)
                        if (k % L == j)
                            for (int i = 0; i < 3; i++)
                                y[i][j] += t[i];
                };
                int k = RS_SLOTS;
                for (int kx = x0; kx < x0 + nx; kx++, k++)
                {
                    const int me = here(lane);
                    const T *x = reinterpret_cast<const T *>(rs_lds + cx[kx * SLICE + me]);
                    const T *w = mx + 9 * kx * SLICE + me;
                    T t[3];
                    for (int i = 0; i < 3; i++)
                        t[i] = block<REF>(w[(3 * i) * SLICE], w[(3 * i + 1) * SLICE],
                                          w[(3 * i + 2) * SLICE], x[0], x[1], x[2]);
                    add(k, t);
                }
#pragma clang loop unroll(disable)
                for (; k < ws; k++)
                {
                    const size_t at = (size_t)base + k * SLICE;
                    const T *x = dl + 3 * (int)glob(rb.pos)[at + here(lane)];
                    const G<T> *w = glob(Vecs<T>::W(d)) + 9 * at + here(lane);
                    T t[3];
                    for (int i = 0; i < 3; i++)
                        t[i] = block<REF>(w[(3 * i) * SLICE], w[(3 * i + 1) * SLICE],
                                          w[(3 * i + 2) * SLICE], x[0], x[1], x[2]);
                    add(k, t);
                }
                for (int i = 0; i < 3; i++)
                    q[i] = phases<L>(y[i]);
            }
            publish(slice_sum<L>(block_row<double>((double)dv[0], (double)dv[1], (double)dv[2],
                                                   (double)q[0], (double)q[1], (double)q[2])),
                    64, 1, words_dq, sm_dq);
            gather(1, words_dq, sm_dq, false);
            if (!meet())
            {
                failed = true;
                break;
            }
            double sq[1];
            total(sm_dq, sq);
            const double dq = sq[0];
            if (REF ? dq == 0.0 || !isfinite(dq) : !(dq > 0.0) || !isfinite(dq))
            {
                // d.Wd == 0 (BaraffCloth.cpp:547-551), or, to a tolerance, a
                // loss of definiteness: stop after a final true residual
                if (tid == 0)
                {
                    sh_st.final_check = 1;
                    sh_st.breakdown = dq == 0.0 ? 0 : 1;
                }
                check = due = true;
                continue;
            }
            // k_cg_update
            const double alpha = uniform(rho / dq);
            double v[2] = {0.0, 0.0};
            for (int i = 0; i < 3; i++)
            {
                if constexpr (MIXED)
                    x32[i] = x32[i] + (float)(alpha * (double)dv[i]);
                else
                    x64[i] = fma_t(alpha, (double)dv[i], x64[i]);
                r[i] = (T)fma_t(-alpha, (double)q[i], (double)r[i]);
                z[i] = P[i] * r[i];
                v[0] = fma_t((double)r[i], (double)z[i], v[0]);
                v[1] = fma_t((double)r[i], (double)r[i], v[1]);
            }
            ++tag;
            publish_z();
            publish(wave_sum2(v[0], v[1]), 32, 2, words_rz, sm_rz);
            gather(2, words_rz, sm_rz, true);
            if (!meet())
            {
                failed = true;
                break;
            }
            double t[2];
            total(sm_rz, t);
            rz = t[0];
            rr = t[1];
            steps++;
            first = false;
            if constexpr (!MIXED)
                if (steps % PROGRESS == 0 && pt.slice0 == pt.set0 && tid == 0)
                    atomicAdd(&a.ctl->progress, 1);
            // (NaN and infinity too)
            check = (steps >= room) | (!REF && !(rr > enough && rr < __builtin_inf()));
        }
        if (failed)
        {
            if (tid == 0 && (!MIXED || a.give_up >= 0 || sh_failed))
                __hip_atomic_store(&a.ctl->aborted, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            else if (tid == 0 && pt.slice0 == pt.set0)
            {
                // on to the FP64 matrix: the launches form this true residual
                // again and go on from it
                CgState st = sh_st;
                st.start = st.first = 1;
                st.updates -= 1;
                store_state(glob(d.cg) + 2 * inst, st);
                store_state(glob(d.cg) + 2 * inst + 1, st);
                rb.epoch[inst] = tag;
            }
            return;
        }
        // the solution and the state for k_update_positions and the host, or
        // what a paused solve goes on with
        if (PAUSE && paused)
        {
            if (have)
                for (int i = 0; i < 3; i++)
                {
                    glob(Vecs<T>::r(d))[3 * row() + i] = r[i];
                    glob(Vecs<T>::d0(d))[3 * row() + i] = dv[i];
                    if constexpr (MIXED)
                        glob(d.dx32)[3 * row() + i] = x32[i];
                    else
                        glob(d.dx)[3 * row() + i] = x64[i];
                }
        }
        else if (have)
            for (int i = 0; i < 3; i++)
            {
                if constexpr (MIXED)
                    glob(d.dx32)[3 * row() + i] = 0.0f;
                else
                    glob(d.dx)[3 * row() + i] = x64[i];
            }
        if (pt.slice0 == pt.set0 && tid == 0)
        {
            CgState st = sh_st;
            st.rho = rho;
            st.first = first;
            if (PAUSE && paused)
            {
                st.since = steps;
                st.rr = rr;
                st.rr_true = rz;
            }
            st.iter = st.total;
            store_state(glob(d.cg) + 2 * inst, st);
            store_state(glob(d.cg) + 2 * inst + 1, st);
            rb.epoch[inst] = tag;
        }
    }
}

__global__ void k_cg_restart(CgState *st, const InstParams *params, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    CgState z = {};
    z.start = 1;
    z.first = 1;
    z.stalls = st[2 * i].stalls;
    z.w64 = z.stalls >= params[i].carry ? 1 : 0;
    st[2 * i] = z;
    st[2 * i + 1] = z;
}

using ResidentKernel = void (*)(ResidentLaunch);

template <int L, bool PAUSE = false> ResidentKernel kernel_for(bool fp32)
{
    return fp32 ? k_resident<float, RS_WAVES32, L, false, PAUSE>
                : k_resident<double, RS_WAVES64, L, false, PAUSE>;
}

// lpr 0: the reference's semantics
ResidentKernel kernel_of(bool fp32, int lpr, bool pause)
{
    if (pause)
        return kernel_for<1, true>(fp32);
    if (lpr == 0)
        return k_resident<double, RS_WAVES64, 1, true>;
    return lpr == 1 ? kernel_for<1>(fp32) : lpr == 2 ? kernel_for<2>(fp32) : kernel_for<4>(fp32);
}

} // namespace

size_t resident_lds(bool fp32, int sets_max, int halo_max, int extra)
{
    static_assert(3 * sizeof(float) * (resident_slices(true) * SLICE + RS_HALO32) < 65536 &&
                      3 * sizeof(double) * (resident_slices(false) * SLICE + RS_HALO64) < 65536,
                  "16-bit offsets into the directions");
    const size_t entries = (size_t)resident_slices(fp32) * SLICE + halo_max;
    return 4 * sizeof(double) * (size_t)sets_max +
           entries * 3 * (sizeof(double) + (fp32 ? sizeof(float) : sizeof(double))) +
           sizeof(int) * (size_t)halo_max + resident_slot_bytes(fp32) * (size_t)extra;
}

int resident_capacity(bool fp32, int lpr, size_t lds, bool pause)
{
    const void *k = reinterpret_cast<const void *>(kernel_of(fp32, lpr, pause));
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        // (the same limit from every thread: the attribute is the process's)
        hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)RS_LDS_MAX) !=
            hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, resident_slices(fp32) * SLICE,
                                                     lds) != hipSuccess)
    {
        (void)hipGetLastError();
        return 0;
    }
    return cus * per_cu;
}

void launch_resident(const ResidentLaunch &a, bool fp32, int grid, hipStream_t s)
{
    hipLaunchKernelGGL(kernel_of(fp32, a.lpr, a.pause > 0), dim3(grid),
                       dim3(resident_slices(fp32) * SLICE),
                       resident_lds(fp32, a.sets_max, a.halo_max, a.extra), s, a);
}

void launch_cg_restart(const DeviceBatch &d, hipStream_t s)
{
    hipLaunchKernelGGL(k_cg_restart, dim3((d.n_inst + 63) / 64), dim3(64), 0, s, d.cg, d.params,
                       d.n_inst);
}

} // namespace bw
