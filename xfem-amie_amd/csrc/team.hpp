// The CG of one problem by a team of workgroups that keep it on the chip.
//
// The launch path streams every vector of the iteration through HBM and ends
// each phase with a kernel boundary: on the 512-RVE batch the vectors are 60 %
// of an iteration's bytes, on a single mesh the three launches and their gaps
// are 15-20 us an iteration whatever its size.  Here a problem is cut into
// groups of tiles, one workgroup of 512 threads (one CU) each; the workgroups
// of a problem (its team) run the whole solve in one launch:
//   - y, r and q of a thread's rows stay in registers, p of the workgroup's
//     rows and of its halo (the rows of other members that its matrix columns
//     name) in LDS.  An iteration reads the matrix (from L2 / MALL after the
//     first) and a 16-bit local column per block, and no vector.
//   - one exchange an iteration: a member publishes the partial sums of its
//     tiles and q of the rows that others' halos hold, waits for everybody's,
//     and then every member computes the same scalars from the same sums.  A
//     reader keeps r and p of its halo up to date by itself (r -= alpha q,
//     p = M r + beta p, the owner's own operations on the owner's numbers), so
//     the exchange of q replaces the one of p and the second wait that it
//     would need.
// Exchanged values travel as 8-byte words {32 bits of the value, 32-bit
// sequence number}, stored and polled with relaxed agent-scope atomics: the
// number says that the value has arrived, so no fence (an L2 write-back on
// CDNA's non-coherent XCD L2s) and no counter stands between members.  An
// all-to-all exchange of this kind takes 1.1 us among 2-8 workgroups, 2 us
// among 64 and 2.5-3.5 us among 256 (a grid barrier with agent-scope fences:
// 2.2 us among 64, 7.4 among 256, before any data is read).  Two buffers
// alternate: a member overwrites a number two exchanges later, when every
// member's sums of the exchange between have told it that they were read.
// The sums of a tile, and of a problem's tiles, are formed in the order of the
// launch path (wg_sum_all, problem_sums2), and every row runs its operations:
// the results are the launch path's bit for bit.
//
// A refinement (every ~100 iterations) publishes x64 through global memory
// with agent-scope fences, recomputes the residual from the FP64 planes and
// exchanges r of the halo rows.
//
// Measured on an MI355X, microseconds an iteration, launch path -> team: P1
// 16^2 FP64 18.2 -> 2.4, P1 128^2 FP64 16.5 -> 4.5, P2 45^2 FIX48 20 -> 6.7, Tet4
// 19^3 block Jacobi 21 -> 8.2, P2 250^2 40 -> 13.4, 64 RVEs of 32..256 cells
// with three loads 100 -> 48 (value-indexed) and 110 -> 71 (planes), Tet4 64^3
// 62 -> 48, P2 400^2 61 -> 42.  What bounds it: on small problems the dependent
// chain of one iteration (product, transposing sums, one exchange of 1.5 us,
// scalars, update); on large ones the latency of the matrix stream at 8
// wavefronts a CU (P2 400^2 reads 106 MB an iteration at 2.4 TB/s, Tet4 64^3 132
// at 2.7, a copy runs at 6.3; wavefronts wait 58-66 % of their cycles), the
// members' halo words, and the spread of the members' times, which the exchange
// waits for.  Where that makes launches faster they run (team.hip).
//
// The workgroups of a launch (at most one per CU, launched cooperatively, so
// all are resident) claim members in a fixed order from a counter, all
// members of a problem in a row; a finished workgroup claims the next.  A
// team waits only for members that resident workgroups will claim, so every
// wait ends; a wait that sees neither its data nor any team's progress for
// seconds gives up and ends the launch.  Its workgroup may publish sums of
// what it did not get until its period ends, but the error flag is visible
// before they are, and is looked at before a refinement: x64 only ever holds
// refinements of valid iterates, a problem converges by their residuals only,
// and the host finishes the others by launches.
#pragma once
#include "device.hpp"

namespace amie {

// 512 threads with 256 registers each: at 1024 with 128 the rows' state left the
// compiler to spill (the update alone took 38 us for 32 slices, 512 RVE sizes)
constexpr int TEAM_WG = 512;
constexpr int TEAM_WAVES = TEAM_WG / WAVE;
constexpr int TEAM_COLS = WG;       // column sums of a problem's tiles (problem_sums2 runs WG threads)

struct TeamMember {
    int32_t prob, m, G;             // problem, member of G
    int32_t nsl;                    // local slices: 4 per tile of the member
    int32_t sl0, mt0;               // its ranges of TeamArgs::mslice and mtile
    int32_t tile0, ntiles;          // the problem's tiles
    int32_t halo0, nhalo;           // its range of TeamArgs::halo
    int64_t xb;                     // the problem's exchange buffer, in 16-byte entries
};

struct TeamArgs {
    const TeamMember *members;
    const int32_t *order;           // members in the order they are claimed
    int32_t nitems;
    int32_t max_periods;            // checkpoint periods per problem
    int32_t ce;                     // iterations per checkpoint period
    int32_t dict_n;                 // entries of the value-indexed matrix's table (copied to LDS)
    const int32_t *mslice;          // local slice -> slice (-1: the tile has fewer)
    const int32_t *mtile;           // local tile -> tile of the problem
    const uint16_t *lidx;           // per slot: own local row, or own rows + halo entry
    const uint32_t *halo;           // global rows of the halos
    const uint8_t *exported;        // per row: some other member's halo holds it
    uint64_t *xb;                   // tile sums: two words per value
    uint64_t *ql[2], *qh[2];        // q / r of exported rows by parity: low words, high words (FP64)
    uint32_t seq0;                  // sequence numbers of earlier passes are at most this
    uint32_t *ctl;                  // [0] ticket, [1] progress, [2] error, [3] largest sequence number used
};

__device__ inline void team_store(uint64_t *p, uint32_t v, uint32_t seq)
{
    __hip_atomic_store(p, ((uint64_t)seq << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline uint64_t team_load(const uint64_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline bool team_is(uint64_t w, uint32_t seq) { return (uint32_t)(w >> 32) == seq; }

// A value of the working precision as one (float) or two (double) words.
template <typename W> struct TeamWord;
template <> struct TeamWord<float> {
    __device__ static inline void store(uint64_t *l, uint64_t *, size_t i, float v, uint32_t seq)
    {
        team_store(l + i, __float_as_uint(v), seq);
    }
    uint64_t a;
    __device__ inline void load(const uint64_t *l, const uint64_t *, size_t i) { a = team_load(l + i); }
    __device__ inline bool is(uint32_t seq) const { return team_is(a, seq); }
    __device__ inline float value() const { return __uint_as_float((uint32_t)a); }
};
template <> struct TeamWord<double> {
    __device__ static inline void store(uint64_t *l, uint64_t *h, size_t i, double v, uint32_t seq)
    {
        team_store(l + i, (uint32_t)__double2loint(v), seq);
        team_store(h + i, (uint32_t)__double2hiint(v), seq);
    }
    uint64_t a, b;
    __device__ inline void load(const uint64_t *l, const uint64_t *h, size_t i)
    {
        a = team_load(l + i);
        b = team_load(h + i);
    }
    __device__ inline bool is(uint32_t seq) const { return team_is(a, seq) && team_is(b, seq); }
    __device__ inline double value() const { return __hiloint2double((int)(uint32_t)b, (int)(uint32_t)a); }
};

// One wait: polls counted, and every few thousand the clock.  It gives up
// (returns false) when another workgroup did, or when neither its data nor
// any team's progress was seen for TEAM_PATIENCE ticks of the 100 MHz clock:
// a member may wait for a peer that still works on an earlier problem, which
// moves the progress count at every checkpoint period.
constexpr long long TEAM_PATIENCE = 500000000ll;   // 5 s
struct TeamWait {
    uint32_t polls = 0, seen = 0;
    long long since = 0;
    __device__ inline bool again(uint32_t *ctl)
    {
        __builtin_amdgcn_s_sleep(1);
        if (++polls & 4095u) return true;
        if (__hip_atomic_load(ctl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return false;
        const uint32_t pr = __hip_atomic_load(ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const long long now = wall_clock64();
        if (since == 0 || pr != seen) {
            since = now;
            seen = pr;
            return true;
        }
        if (now - since < TEAM_PATIENCE) return true;
        __hip_atomic_store(ctl + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0);   // before anything that follows
        return false;
    }
};

// ------------------------------------------------ sums over a wavefront
// The xor butterfly of wave_sum (32, 16, 8, 4, 2, 1) on N values at once:
// while more than one value is left, a step adds two of them in one exchange,
// the lanes with the step's bit clear going on with the first and the others
// with the second.  The additions of each value are wave_sum's (a butterfly's
// partners hold the same partial sums), with N + 4 or so exchanges instead of
// 6 N, none through LDS (the swaps of gfx950 and DPP moves).
template <int CTRL> __device__ inline double dpp_move(double v)
{
    // every lane of these patterns has a source: the old value is never seen
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}
// the value of lane ^ MASK, MASK <= 8: a rotation by half a row of 16 lanes,
// two mirrors, two quad permutations
template <int MASK> __device__ inline double lane_xor(double v)
{
    if constexpr (MASK == 8) return dpp_move<0x128>(v);
    else if constexpr (MASK == 4) return dpp_move<0x1B>(dpp_move<0x141>(v));
    else if constexpr (MASK == 2) return dpp_move<0x4E>(v);
    else return dpp_move<0xB1>(v);
}
// a of a lane and its partner's in lanes with MASK clear, b's in the others
template <int MASK> __device__ inline double pair_sum(double a, double b, int lane)
{
    if constexpr (MASK >= 16) {
        const uint32_t al = (uint32_t)__double2loint(a), ah = (uint32_t)__double2hiint(a);
        const uint32_t bl = (uint32_t)__double2loint(b), bh = (uint32_t)__double2hiint(b);
        if constexpr (MASK == 32) {
            const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
            const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
            return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
        } else {
            const auto l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
            const auto h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
            return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
        }
    } else {
        const bool up = (lane & MASK) != 0;
        return (up ? b : a) + lane_xor<MASK>(up ? a : b);
    }
}
template <int N, int MASK> struct WaveFold {
    static constexpr int H = N / 2, NN = H + N % 2;
    __device__ static inline void run(double *v, int *id, int lane)
    {
        const int up = (lane & MASK) ? -1 : 0;
#pragma unroll
        for (int i = 0; i < H; i++) {
            v[i] = pair_sum<MASK>(v[2 * i], v[2 * i + 1], lane);
            // by bits: a choice between two array entries goes through memory
            id[i] = id[2 * i] ^ ((id[2 * i] ^ id[2 * i + 1]) & up);
        }
        if constexpr (N % 2) {
            v[H] = pair_sum<MASK>(v[N - 1], v[N - 1], lane);
            id[H] = id[N - 1];
        }
        if constexpr (MASK > 1) WaveFold<NN, MASK / 2>::run(v, id, lane);
    }
};
// Sums v[0..N) over the wavefront (v is used up); returns the sum of value
// `id`, which differs by lane: lane ^ 1 always holds the same.  N <= 32.
template <int N> __device__ inline double wave_sums(double *v, int lane, int &id)
{
    static_assert(N <= 32, "one value per pair of lanes");
    int ids[N];
#pragma unroll
    for (int i = 0; i < N; i++) ids[i] = i;
    WaveFold<N, 32>::run(v, ids, lane);
    id = ids[0];
    return v[0];
}

// ------------------------------------------------------ blocks of a row
// Matrix blocks by ordinary (cached) loads: from the second iteration on they
// come from L2 or the MALL.  The slot is a wavefront-uniform base (a scalar
// address) and a lane.
template <typename M, int B> struct TeamBlk;
template <int B> struct TeamBlk<Pre64, B> {
    static constexpr int NP = B * B / 2;
    d2v p[NP];
    double rem;
    __device__ inline void load(const void *base, int64_t ns, int64_t s0, int lane)
    {
        const d2v *q = reinterpret_cast<const d2v *>(base) + s0;
#pragma unroll
        for (int i = 0; i < NP; i++) p[i] = (q + i * ns)[lane];
        if constexpr (B * B % 2) rem = (reinterpret_cast<const double *>(reinterpret_cast<const d2v *>(base) + NP * ns) + s0)[lane];
    }
    __device__ inline double at(const double *, int k) const
    {
        if constexpr (B * B % 2) {
            if (k == B * B - 1) return rem;
        }
        return k % 2 ? p[k / 2].y : p[k / 2].x;
    }
    __device__ inline void keep() {}
};
template <int B> struct TeamBlk<Fix48, B> {
    typename BlkRaw<Fix48, B>::Raw r;
    __device__ inline void load(const void *base, int64_t ns, int64_t s0, int lane)
    {
        const u4v *q = reinterpret_cast<const u4v *>(base);
        const char *c = reinterpret_cast<const char *>(base);
        if constexpr (B == 2) {
            r.l = (q + s0)[lane];
            r.h = (reinterpret_cast<const u2v *>(c + ns * 16) + s0)[lane];
        } else {
            r.l0 = (q + s0)[lane];
            r.l1 = (q + ns + s0)[lane];
            r.l2 = (reinterpret_cast<const uint32_t *>(q + 2 * ns) + s0)[lane];
            r.h0 = (reinterpret_cast<const u4v *>(c + ns * 36) + s0)[lane];
            r.h1 = (reinterpret_cast<const uint16_t *>(c + ns * 52) + s0)[lane];
        }
    }
    __device__ inline double at(const double *, int k) const { return BlkRaw<Fix48, B>::at(r, k); }
    __device__ inline void keep()
    {
        if constexpr (B == 2) asm volatile("" : "+v"(r.l), "+v"(r.h));
        else asm volatile("" : "+v"(r.l0), "+v"(r.l1), "+v"(r.l2), "+v"(r.h0), "+v"(r.h1));
    }
};
template <int B> struct TeamBlk<Dict, B> {
    uint32_t id;
    __device__ inline void load(const void *base, int64_t, int64_t s0, int lane)
    {
        id = (reinterpret_cast<const uint16_t *>(base) + s0)[lane];
    }
    __device__ inline double at(const double *tab, int k) const { return tab[id * DictEntry<B>::N + k]; }
    __device__ inline void keep() { asm volatile("" : "+v"(id)); }
};

// A group of N blocks of a row.
template <typename M, int B, int N> struct TeamGroup {
    uint32_t li[N];
    TeamBlk<M, B> blk[N];
    // blocks from slot s0 on, `left` of them in the row: past it the null
    // slots (zero blocks), so that no branch stands between the loads
    __device__ inline void load(const uint16_t *lidx, const void *vals, int64_t ns, int64_t s0, int left, int lane)
    {
        int64_t s[N];
#pragma unroll
        for (int u = 0; u < N; u++) s[u] = u < left ? s0 + u * WAVE : ns - WAVE;
#pragma unroll
        for (int u = 0; u < N; u++) li[u] = (lidx + s[u])[lane];
#pragma unroll
        for (int u = 0; u < N; u++) blk[u].load(vals, ns, s[u], lane);
    }
};

// The first blocks of a thread's rows stay in registers for the whole solve
// and the rest of a longer row is streamed: as many blocks, in quads, as the
// registers beside the rows' state take without spilling.  (Products of 7
// blocks a row: 2600 -> 1700 cycles of an iteration.  3 x 3 blocks are too
// large, more than two slices a wavefront too many; of the value-indexed
// matrix a block is one register.)
template <typename M, int B, int NR, int J> constexpr int team_resident()
{
    if (std::is_same<M, Dict>::value) return J * NR * B <= 8 ? 8 : 0;
    if (B == 3 || J > 2) return 0;
    if (NR == 3) return J == 1 ? 8 : 0;
    return J == 2 ? 8 : (std::is_same<M, Fix48>::value ? 16 : 12);
}
template <typename M, int B, int R> struct TeamRes {
    uint32_t li[R / 2];   // two local columns a register
    TeamBlk<M, B> blk[R];
    __device__ inline void load(const uint16_t *lidx, const void *vals, int64_t ns, int64_t s0, int width, int lane)
    {
#pragma unroll
        for (int u = 0; u < R; u++) {
            const int64_t s = u < width ? s0 + u * WAVE : ns - WAVE;
            const uint32_t l = (lidx + s)[lane];
            li[u / 2] = u % 2 ? li[u / 2] | l << 16 : l;
            blk[u].load(vals, ns, s, lane);
        }
    }
    // Said to change each iteration: addresses and values made from them are
    // then made again, not kept beside them in registers that spill.
    __device__ inline void keep(int u0)
    {
#pragma unroll
        for (int u = u0; u < u0 + 4; u++) {
            if (u % 2 == 0) asm volatile("" : "+v"(li[u / 2]));
            blk[u].keep();
        }
    }
    __device__ inline uint32_t col(int u) const { return u % 2 ? li[u / 2] >> 16 : li[u / 2] & 0xffffu; }
};
template <typename M, int B> struct TeamRes<M, B, 0> {
    __device__ inline void load(const uint16_t *, const void *, int64_t, int64_t, int, int) {}
};

// A row's NR x B values (p in LDS, the exchanged words): one record per row,
// right-hand sides next to each other, so a gather is one address.  (Records
// of 24 bytes for consecutive rows are free of bank conflicts.)
template <typename W, int B, int NR> __device__ inline void rec_load(const W *p, W (*o)[B])
{
    if constexpr (B == 2) {
        typedef W v2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const v2 t = reinterpret_cast<const v2 *>(p)[k];
            o[k][0] = t.x;
            o[k][1] = t.y;
        }
    } else {
#pragma unroll
        for (int k = 0; k < NR; k++)
#pragma unroll
            for (int i = 0; i < B; i++) o[k][i] = p[k * B + i];
    }
}
template <typename W, int B, int NR> __device__ inline void rec_store(W *p, const W (*o)[B])
{
    if constexpr (B == 2) {
        typedef W v2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int k = 0; k < NR; k++) {
            v2 t;
            t.x = o[k][0];
            t.y = o[k][1];
            reinterpret_cast<v2 *>(p)[k] = t;
        }
    } else {
#pragma unroll
        for (int k = 0; k < NR; k++)
#pragma unroll
            for (int i = 0; i < B; i++) p[k * B + i] = o[k][i];
    }
}

// the row's inverse diagonal block, by ordinary loads
template <typename W, int B, bool BJ> __device__ inline void team_minv(const void *minv, int row, W *mi)
{
    if constexpr (BJ) {
        const W *m = cvw<W>(minv) + (size_t)row * (B * B);
#pragma unroll
        for (int k = 0; k < B * B; k++) mi[k] = m[k];
    }
}

// LDS of a member beside the table: p of own rows and halo, r of the halo.
inline size_t team_lds(int64_t rows_and_twice_halo, int b, int nr, int word)
{
    return (size_t)nr * b * word * (size_t)rows_and_twice_halo;
}

// The kernel's arguments, read again from the kernel argument segment where a
// phase needs them (args() hides the pointer from the compiler): kept in
// scalar registers over the iteration they would spill, and the addresses
// formed from them would be hoisted into vector registers.
struct TeamAll {
    SolveArgs a;
    TeamArgs t;
};
// (KEEP: with one slice a wavefront and no resident blocks there is room.)
typedef const __attribute__((address_space(4))) TeamAll *TeamPtr;
template <bool KEEP> __device__ inline TeamPtr team_args_of()
{
    TeamPtr p = (TeamPtr)__builtin_amdgcn_kernarg_segment_ptr();
    if (!KEEP) asm volatile("" : "+s"(p));
    return p;
}

// lane k's value in every lane
__device__ inline double lane_value(double v, int k)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), k), __builtin_amdgcn_readlane(__double2loint(v), k));
}

__device__ inline double lane_at(double v, int k) { return lane_value(v, __builtin_amdgcn_readfirstlane(k)); }

// J: slices per wavefront (wavefront w has the local slices w, w + 8, ...).
// Registers: y, r, q of J rows, NR B (8 + 2 sizeof(W)) bytes each.
template <typename W, typename M, int B, int NR, bool BJ, int J>
__global__ __launch_bounds__(TEAM_WG) void k_cg_team(TeamAll all_)
{
    // exchanged values: K1's sums, r.z (= r.r without block Jacobi), r.r,
    // and after a refinement the two FP64 residual norms
    constexpr int NRES = BJ ? 2 * NR : NR;
    constexpr int NVN = 3 * NR + NRES, NVC = NVN + 2 * NR;
    constexpr int MAXT = TEAM_WAVES * J / TILE_SLICES;   // tiles of a member
    constexpr int MAXV = (NVC + TEAM_WAVES - 1) / TEAM_WAVES;   // values per wavefront
    constexpr int NGRP = TEAM_COLS / WAVE;
    constexpr int NDIR = NR == 1 ? NGRP : 1;   // groups of 64 tiles summed in one step
    constexpr int REC = NR * B;
    static_assert(MAXT <= 16 && NVC * 16 <= TEAM_WG, "one thread per tile and value");
    extern __shared__ __align__(16) char dyn[];
    __shared__ ProbDev P;
    __shared__ int4 sdesc[TEAM_WAVES * J];                // slot pointer lo, hi, width | rows << 16, slice
    __shared__ double wsum[TEAM_WAVES * J][3 * NR];       // sums of a slice: K1's,
    __shared__ double wres[2][TEAM_WAVES * J][NVC - 3 * NR];   // the residual's (two buffers)
    __shared__ double grp[TEAM_WAVES / NGRP][NGRP];       // sums of 64 columns
    __shared__ double red_[TEAM_WAVES][NVC];              // sums of the problem (a team of one: per wavefront)
    __shared__ int s_item, s_bad;
    (void)all_;
    constexpr bool KEEP = J == 1 && team_resident<M, B, NR, J>() == 0;
    constexpr auto team_args = team_args_of<KEEP>;
    const int wave = wave_id();
    int lane = threadIdx.x % WAVE, tid = threadIdx.x;
    // Said to change, so that lane masks made from them are made where they
    // are used: kept over the iteration they fill the scalar registers, and
    // what spills there is read back a lane at a time.
    // (Measured: 3 % of P1 128^2, the other way by as much where a row has
    // more values and the scalar work hides.)
    auto fresh = [&] {
        if (B == 2 && NR == 1) asm volatile("" : "+v"(lane), "+v"(tid));
    };
    size_t tab_bytes = 0;
    if constexpr (std::is_same<M, Dict>::value) {
        TeamPtr A = team_args();
        const int nd = A->t.dict_n * DictEntry<B>::N;
        for (int i = tid; i < nd; i += TEAM_WG) reinterpret_cast<double *>(dyn)[i] = A->a.dict_table[i];
        tab_bytes = (size_t)nd * 8;
    }
    const double *tab = reinterpret_cast<const double *>(dyn);
    W *lp = reinterpret_cast<W *>(dyn + tab_bytes);
    if (tid == 0) s_bad = 0;
    uint32_t seq_max = team_args()->t.seq0;
    for (;;) {
        __syncthreads();   // the last problem's LDS is free
        if (tid == 0)
            s_item = (int)__hip_atomic_fetch_add(team_args()->t.ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const int item = __builtin_amdgcn_readfirstlane(s_item);
        TeamPtr A0 = team_args();
        if (item >= A0->t.nitems || s_bad) break;
        const TeamMember mb = A0->t.members[A0->t.order[item]];
        ProbDev *const gP = A0->a.prob + mb.prob;
        if (gP->status != ST_RUNNING) continue;
        for (int i = tid; i < (int)(sizeof(ProbDev) / 4); i += TEAM_WG)
            reinterpret_cast<uint32_t *>(&P)[i] = reinterpret_cast<const uint32_t *>(gP)[i];
        const int G = mb.G, rows = mb.nsl * WAVE, H = mb.nhalo;
        const int mytiles = mb.nsl / TILE_SLICES;
        const bool hop = mb.ntiles > NDIR * WAVE;   // the sums take two steps (collect)
        W *lr = lp + REC * (rows + H);         // r of the halo
        uint32_t xs = A0->t.seq0, qs = xs;     // sequence numbers of the sums and of the rows
        uint64_t *const xbase = A0->t.xb + 2 * mb.xb;
        auto xb_at = [&](uint32_t seq, int v, int t) { return xbase + 2 * (((seq & 1) * NVC + v) * mb.ntiles + t); };
        auto total_at = [&](uint32_t seq, int v) { return xbase + 2 * (2 * NVC * mb.ntiles + (seq & 1) * NVC + v); };
        // this thread's tile and value of a publication, and its first halo row
        const int pt = tid & 15, pv = (NR == 1 ? TEAM_WG - 1 - tid : tid) >> 4;
        const int ptile = pt < mytiles ? A0->t.mtile[mb.mt0 + pt] : 0;
        const int halo_row = tid < H ? (int)A0->t.halo[mb.halo0 + tid] : 0;
        if (tid < TEAM_WAVES * J) {
            const int gl = tid < mb.nsl ? A0->t.mslice[mb.sl0 + tid] : -1;
            const int4 sd = A0->a.slice_desc[gl < 0 ? 0 : gl];
            sdesc[tid] = gl < 0 ? make_int4(0, 0, 0, 0) : make_int4(sd.x, sd.y, sd.z | sd.w << 16, gl);
        }
        for (int i = tid; i < REC * (rows + H); i += TEAM_WG) lp[i] = 0;
        __syncthreads();
        // slice j of this wavefront, from LDS
        struct Slice {
            int64_t s0;
            int width, row;
            bool own;
        };
        auto slice = [&](int j) {
            const int4 d = sdesc[wave + j * TEAM_WAVES];
            const int wr = __builtin_amdgcn_readfirstlane(d.z);
            Slice s;
            s.s0 = (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane(d.x) |
                   ((int64_t)__builtin_amdgcn_readfirstlane(d.y) << 32);
            s.width = wr & 0xffff;
            s.row = __builtin_amdgcn_readfirstlane(d.w) * WAVE + lane;
            s.own = lane < (wr >> 16);
            return s;
        };
        const Slice first_slice = slice(0);
        auto slice_of = [&](int j) { return J == 1 ? first_slice : slice(j); };
        uint32_t expo = 0;   // bit j: the row of slice j is exported
        double y[J][NR][B];
        W r[J][NR][B], q[J][NR][B];
#pragma unroll
        for (int j = 0; j < J; j++) {
            const Slice s = slice(j);
            if (s.own && G > 1 && A0->t.exported[s.row]) expo |= 1u << j;
#pragma unroll
            for (int k = 0; k < NR; k++)
#pragma unroll
                for (int i = 0; i < B; i++) {
                    y[j][k][i] = 0.;
                    r[j][k][i] = q[j][k][i] = 0;
                }
        }
        W hv[NR][B];   // the thread's first halo row, as collected

        // Sums of N values of the wavefront's slice j into wsum, from value vfirst on.
        // (The residual's: r.z is still read by slow wavefronts of a team of one
        // when the next update writes it.)
        int rp = 0;
        auto slice_sums = [&](double *v, auto n, int vfirst, int j) {
            constexpr int N = decltype(n)::value;
            int id;
            const double s = wave_sums<N>(v, lane, id);
            double *to = vfirst < 3 * NR ? &wsum[wave + j * TEAM_WAVES][vfirst]
                                         : &wres[rp][wave + j * TEAM_WAVES][vfirst - 3 * NR];
            if ((lane & 1) == 0) to[id] = s;
        };
        auto tile_sum = [&](int t, int v) {
            const bool k1 = v < 3 * NR;
            const int ld = k1 ? 3 * NR : NVC - 3 * NR;
            const double *l = k1 ? &wsum[t * TILE_SLICES][v] : &wres[rp][t * TILE_SLICES][v - 3 * NR];
            return (l[0] + l[ld]) + (l[2 * ld] + l[3 * ld]);
        };
        double *const red = red_[G == 1 ? wave : 0];
        auto put_sum = [&](uint64_t *o, double s, uint32_t seq) {
            team_store(o, (uint32_t)__double2loint(s), seq);
            team_store(o + 1, (uint32_t)__double2hiint(s), seq);
        };
        auto poll_sum = [&](const uint64_t *o, uint32_t seq, double &v) {
            TeamWord<double> w;
            w.load(o, o + 1, 0);
            v = w.value();
            return w.is(seq);
        };
        // Tile sums of values [v0, v1) from wsum, published with number seq
        // (a team of one reads them there).
        auto publish = [&](int v0, int v1, uint32_t seq) {
            const int v = v0 + pv;
            if (G > 1 && pt < mytiles && v < v1) put_sum(xb_at(seq, v, ptile), tile_sum(pt, v), seq);
        };
        // A row's words.  A poll issues every load before it looks at one (a
        // wait is for one trip of 900 cycles then, not for one a word), so
        // lanes with nothing to read read word 0 and ignore it.
        struct Row {
            TeamWord<W> w[NR * B];
            __device__ inline void load(TeamPtr A, uint32_t seq, int gr)
            {
                const uint64_t *ql = A->t.ql[seq & 1], *qh = A->t.qh[seq & 1];
#pragma unroll
                for (int i = 0; i < NR * B; i++) w[i].load(ql, qh, (size_t)gr * REC + i);
            }
            __device__ inline bool get(uint32_t seq, W(*v)[B]) const
            {
                bool all = true;
#pragma unroll
                for (int i = 0; i < NR * B; i++) {
                    all &= w[i].is(seq);
                    v[i / B][i % B] = w[i].value();
                }
                return all;
            }
        };
        auto poll_row = [&](TeamPtr A, uint32_t seq, int gr, W(*v)[B]) {
            Row w;
            w.load(A, seq, gr);
            return w.get(seq, v);
        };
        // The problem's sums of values [0, nv) in problem_sums2's order: columns
        // of the tiles t, t + 256, ... in order, a butterfly over each 64
        // columns, the four in pairs.  Up to 256 tiles (64 with three
        // right-hand sides, whose words would need 100 registers) every member
        // reads every tile's values; beyond value v is summed by member v % G
        // alone and published once more, a second step of 1.2 us that 64
        // members make good.  The sums end in red, for
        // every wavefront.  hv receives this thread's first halo row with number
        // hseq, when that is not 0: its wait is the same one.  With one
        // right-hand side the last wavefronts publish and the first ones read:
        // loads behind a store wait for its acknowledgement, one counter
        // serves both (with three all of them read).
        auto group_total = [&](double t, int id) {
            // lane's value is group id's sum: the four in pairs
            static_assert(NGRP == 4, "two pairs");
            int at[NGRP];
#pragma unroll
            for (int g = 0; g < NGRP; g++) at[g] = __builtin_ctzll(__ballot(id == g));
            return (lane_at(t, at[0]) + lane_at(t, at[1])) + (lane_at(t, at[2]) + lane_at(t, at[3]));
        };
        double own_total = 0.;   // a team of one: value `lane`
        auto collect = [&](int nv, uint32_t seq, uint32_t hseq) {
            TeamPtr A = team_args();
            const bool mine = hseq != 0 && tid < H, rows_too = __any(mine);
            TeamWait w;
            bool ok = true;
            if (G == 1) {
                // the tiles are here: the butterfly over at most 16 lanes that
                // hold one, by one lane a value; every wavefront for itself,
                // so that no barrier follows
                if (lane < nv) {
                    double t[MAXT];
#pragma unroll
                    for (int i = 0; i < MAXT; i++) t[i] = i < mytiles ? 0. + tile_sum(i, lane) : 0.;
#pragma unroll
                    for (int h = MAXT / 2; h > 0; h >>= 1)   // (0. + t is not -0.: the zeros beyond change nothing)
#pragma unroll
                        for (int i = 0; i < h; i++) t[i] += t[i + h];
                    red[lane] = own_total = t[0];
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                return;
            }
            if (!hop) {
                // wavefront w reads values w, w + 8, ...
                double s[MAXV][NDIR];
                for (;;) {
                    bool all = true;
                    TeamWord<double> w1[MAXV][NDIR];
                    Row row;
                    auto reads = [&](int i, int g) {
                        return wave + i * TEAM_WAVES < nv && g * WAVE < mb.ntiles;
                    };
#pragma unroll
                    for (int i = 0; i < MAXV; i++)
#pragma unroll
                        for (int g = 0; g < NDIR; g++)
                            if (NDIR == 1 || reads(i, g)) {   // (one group: value nv - 1 again, no branch)
                                const uint64_t *o = xb_at(seq, min(wave + i * TEAM_WAVES, nv - 1),
                                                          min(g * WAVE + lane, mb.ntiles - 1));
                                w1[i][g].load(o, o + 1, 0);
                            }
                    if (rows_too) row.load(A, hseq, halo_row);
#pragma unroll
                    for (int i = 0; i < MAXV; i++)
#pragma unroll
                        for (int g = 0; g < NDIR; g++) {
                            s[i][g] = 0.;
                            if (NDIR == 1 || reads(i, g)) {
                                all &= w1[i][g].is(seq);
                                if (g * WAVE + lane < mb.ntiles) s[i][g] = 0. + w1[i][g].value();
                            }
                        }
                    if (rows_too) all &= row.get(hseq, hv) || !mine;
                    if (__all(all)) break;
                    if (!w.again(A->t.ctl)) { ok = false; break; }
                }
                if constexpr (NDIR == 1) {
                    int id;
                    double sv[MAXV];
#pragma unroll
                    for (int i = 0; i < MAXV; i++) sv[i] = s[i][0];
                    const double tot = wave_sums<MAXV>(sv, lane, id);
                    const int v = wave + id * TEAM_WAVES;
                    if ((lane & 1) == 0 && v < nv) red[v] = tot;
                } else {
                    static_assert(MAXV == 1, "one value a wavefront");
                    const int v = wave;
                    if (v < nv) {
                        // (the columns beyond the tiles are zeros: sums of
                        // empty groups are 0. and adding them changes nothing)
                        int id;
                        double tot;
                        if (mb.ntiles <= WAVE) {
                            tot = wave_sums<1>(s[0], lane, id);
                        } else {
                            const double t = wave_sums<NDIR>(s[0], lane, id);
                            tot = group_total(t, id);
                        }
                        if (lane == 0) red[v] = tot;
                    }
                }
                if (!ok) s_bad = 1;
                __syncthreads();
                return;
            }
            // four wavefronts sum a value
            constexpr int HALVES = TEAM_WAVES / NGRP;
            const int half = wave / NGRP, g = wave % NGRP, nu = (mb.ntiles + TEAM_COLS - 1) / TEAM_COLS;
            for (int v0 = mb.m; v0 < nv; v0 += HALVES * G) {
                const int v = v0 + half * G;
                double s = 0.;
                if (v < nv) {
                    constexpr int Q = 8;   // tiles of a column in flight
                    for (int u0 = 0; u0 < nu; u0 += Q) {
                        double c[Q];
                        for (;;) {
                            bool all = true;
                            TeamWord<double> wu[Q];
#pragma unroll
                            for (int u = 0; u < Q; u++)
                                if (u0 + u < nu) {
                                    const uint64_t *o = xb_at(seq, v, min((u0 + u) * TEAM_COLS + g * WAVE + lane, mb.ntiles - 1));
                                    wu[u].load(o, o + 1, 0);
                                }
#pragma unroll
                            for (int u = 0; u < Q; u++) {
                                const bool use = u0 + u < nu && (u0 + u) * TEAM_COLS + g * WAVE + lane < mb.ntiles;
                                all &= wu[u].is(seq) || !use;
                                c[u] = use ? wu[u].value() : 0.;
                            }
                            if (__all(all)) break;
                            if (!w.again(A->t.ctl)) { ok = false; break; }
                        }
#pragma unroll
                        for (int u = 0; u < Q; u++)
                            if (u0 + u < nu) s += c[u];
                    }
                }
                int id;
                const double tot = wave_sums<1>(&s, lane, id);
                if (lane == 0) grp[half][g] = tot;
                __syncthreads();
                if (lane == 0 && g == (NR == 1 ? NGRP - 1 : 0) && v < nv)
                    put_sum(total_at(seq, v), (grp[half][0] + grp[half][1]) + (grp[half][2] + grp[half][3]), seq);
                if (v0 + HALVES * G < nv) __syncthreads();
            }
            for (;;) {
                bool all = true;
                const uint64_t *o = total_at(seq, lane < nv ? lane : 0);
                TeamWord<double> tot;
                Row row;
                if (wave == 0) tot.load(o, o + 1, 0);
                if (rows_too) row.load(A, hseq, halo_row);
                if (wave == 0) {
                    all &= tot.is(seq) || lane >= nv;
                    if (lane < nv) red[lane] = tot.value();
                }
                if (rows_too) all &= row.get(hseq, hv) || !mine;
                if (__all(all)) break;
                if (!w.again(A->t.ctl)) { ok = false; break; }
            }
            if (!ok) s_bad = 1;
            __syncthreads();
        };
        // Words of q (or r) of the exported row of slice j.
        auto export_row = [&](int j, int row, W(*v)[B], uint32_t seq) {
            if (expo >> j & 1) {
                TeamPtr A = team_args();
                uint64_t *ql = A->t.ql[seq & 1], *qh = A->t.qh[seq & 1];
#pragma unroll
                for (int k = 0; k < NR; k++)
#pragma unroll
                    for (int i = 0; i < B; i++)
                        TeamWord<W>::store(ql, qh, (size_t)row * REC + k * B + i, v[k][i], seq);
            }
        };
        // The halo rows' words, handed to use(h, global row, value[NR][B]);
        // `first`: the thread's first row is in hv.
        auto import_rows = [&](uint32_t seq, auto first, auto use) {
            TeamPtr A = team_args();
            int h = tid;
            if constexpr (decltype(first)::value) {
                if (h < H) use(h, halo_row, hv);
                h += TEAM_WG;
            }
            for (; h < H; h += TEAM_WG) {
                const int gr = (int)A->t.halo[mb.halo0 + h];
                W v[NR][B];
                TeamWait w;
                while (!poll_row(A, seq, gr, v))
                    if (!w.again(A->t.ctl)) { s_bad = 1; break; }
                use(h, gr, v);
            }
        };

        // ---- |S b|^2 and |b|^2 (k_rhs_norms, k_norms_final)
#pragma unroll
        for (int j = 0; j < J; j++) {
            const Slice sl = slice_of(j);
            TeamPtr A = team_args();
            double v[2 * NR];
#pragma unroll
            for (int i = 0; i < 2 * NR; i++) v[i] = 0.;
            if (sl.own)
#pragma unroll
                for (int k = 0; k < NR; k++)
#pragma unroll
                    for (int i = 0; i < B; i++) {
                        const double bv = A->a.b64[k * A->a.vplane + (size_t)sl.row * B + i];
                        const double sb = A->a.S[(size_t)sl.row * B + i] * bv;
                        v[k] = mac(sb, sb, v[k]);
                        v[NR + k] = mac(bv, bv, v[NR + k]);
                    }
            slice_sums(v, std::integral_constant<int, 2 * NR>(), 0, j);
        }
        __syncthreads();
        xs++;
        publish(0, 2 * NR, xs);
        collect(2 * NR, xs, 0);
        if (tid == 0) {
            double s[2 * NR];
            for (int i = 0; i < 2 * NR; i++) s[i] = red[i];
            norm_scalars<NR>(P, s);
            P.src_ckpt = 1;
        }
        __syncthreads();

        // ---- a refinement: x64 += S y, y = 0 (k_ckpt_x), then r64 =
        // b - K x64, r = S r64, p = M r + beta p (k_ckpt_r).  The residual
        // sums (value 3 NR on) are published for the exchange after it.
        auto refine = [&](bool first) {
            if (!first) {
#pragma unroll
                for (int j = 0; j < J; j++) {
                    const Slice sl = slice_of(j);
                    TeamPtr A = team_args();
                    if (sl.own) {
                        double sr[B];
                        Node<double, B>::load(A->a.S + (size_t)sl.row * B, sr);
#pragma unroll
                        for (int k = 0; k < NR; k++) {
                            double *x = A->a.x64 + k * A->a.vplane + (size_t)sl.row * B;
                            double xv[B];
                            Node<double, B>::load(x, xv);
#pragma unroll
                            for (int i = 0; i < B; i++) {
                                xv[i] = mac(sr[i], y[j][k][i], xv[i]);
                                y[j][k][i] = 0.;
                            }
                            Node<double, B>::store(x, xv);
                        }
                    }
                }
                if (G > 1) {
                    // every thread's stores have reached L2, one write-back
                    // publishes them; the exchange of one value per tile is
                    // the barrier
                    __builtin_amdgcn_s_waitcnt(0);
                    __syncthreads();
                    xs++;
                    TeamPtr A = team_args();
                    if (tid == 0) {
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
                        for (int t = 0; t < mytiles; t++) put_sum(xb_at(xs, 0, A->t.mtile[mb.mt0 + t]), 0., xs);
                    }
                    TeamWait w;
                    for (int t = tid; t < mb.ntiles; t += TEAM_WG) {
                        double s;
                        while (!poll_sum(xb_at(xs, 0, t), xs, s))
                            if (!w.again(A->t.ctl)) { s_bad = 1; break; }
                    }
                    __syncthreads();
                    if (s_bad) return;
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                } else {
                    __syncthreads();
                }
            }
            const bool restart = P.first || P.refine == 1;
            qs++;
#pragma unroll
            for (int j = 0; j < J; j++) {
                const Slice sl = slice_of(j);
                TeamPtr A = team_args();
                double v[NRES + 2 * NR];
#pragma unroll
                for (int i = 0; i < NRES + 2 * NR; i++) v[i] = 0.;
                double acc[NR][B];
#pragma unroll
                for (int k = 0; k < NR; k++)
#pragma unroll
                    for (int i = 0; i < B; i++) acc[k][i] = 0.;
                for (int kb = 0; kb < sl.width; kb++) {
                    const int64_t s0 = sl.s0 + (int64_t)kb * WAVE;
                    const uint32_t c = (A->a.col + s0)[lane];
                    TeamBlk<Pre64, B> blk;   // the planes of the unscaled K have the same layout
                    blk.load(A->a.v64, A->a.nslots, s0, lane);
                    double xv[NR][B];
#pragma unroll
                    for (int k = 0; k < NR; k++) Node<double, B>::load(A->a.x64 + k * A->a.vplane + (size_t)c * B, xv[k]);
#pragma unroll
                    for (int jj = 0; jj < B; jj++)
#pragma unroll
                        for (int i = 0; i < B; i++) {
                            const double m = blk.at(nullptr, jj * B + i);
#pragma unroll
                            for (int k = 0; k < NR; k++) acc[k][i] = mac(m, xv[k][jj], acc[k][i]);
                        }
                }
                if (sl.own) {
                    W mi[B * B];
                    team_minv<W, B, BJ>(A->a.minv, sl.row, mi);
                    double sr[B];
                    Node<double, B>::load(A->a.S + (size_t)sl.row * B, sr);
                    W *pl = lp + REC * ((wave + j * TEAM_WAVES) * WAVE + lane);
                    W po[NR][B];
                    rec_load<W, B, NR>(pl, po);
#pragma unroll
                    for (int k = 0; k < NR; k++) {
                        const W be = restart ? (W)0 : (W)P.beta[k];
                        double bv[B];
                        Node<double, B>::load(A->a.b64 + k * A->a.vplane + (size_t)sl.row * B, bv);
                        W zv[B];
#pragma unroll
                        for (int i = 0; i < B; i++) {
                            const double r64 = bv[i] - acc[k][i];
                            const double rs = sr[i] * r64;
                            v[NRES + k] = mac(r64, r64, v[NRES + k]);
                            v[NRES + NR + k] = mac(rs, rs, v[NRES + NR + k]);
                            r[j][k][i] = (W)rs;
                        }
                        precond<W, B, BJ>(mi, r[j][k], zv);
#pragma unroll
                        for (int i = 0; i < B; i++) {
                            po[k][i] = mac(be, po[k][i], zv[i]);
                            v[k] = mac((double)r[j][k][i], (double)zv[i], v[k]);
                            if constexpr (BJ) v[NR + k] = mac((double)r[j][k][i], (double)r[j][k][i], v[NR + k]);
                        }
                    }
                    rec_store<W, B, NR>(pl, po);
                }
                export_row(j, sl.row, r[j], qs);
                slice_sums(v, std::integral_constant<int, NRES + 2 * NR>(), 3 * NR, j);
            }
            import_rows(qs, std::false_type(), [&](int h, int gr, W(*rv)[B]) {
                W mi[B * B];
                team_minv<W, B, BJ>(team_args()->a.minv, gr, mi);
                W *pl = lp + REC * (rows + h);
                W po[NR][B];
                rec_load<W, B, NR>(pl, po);
#pragma unroll
                for (int k = 0; k < NR; k++) {
                    const W be = restart ? (W)0 : (W)P.beta[k];
                    W zv[B];
                    precond<W, B, BJ>(mi, rv[k], zv);
#pragma unroll
                    for (int i = 0; i < B; i++) po[k][i] = mac(be, po[k][i], zv[i]);
                }
                rec_store<W, B, NR>(pl, po);
                rec_store<W, B, NR>(lr + REC * h, rv);
            });
            __syncthreads();
            publish(3 * NR, NVC, xs + 1);
        };
        if (!s_bad) refine(true);

        // streamed groups: 16-37 registers, twice (the next group is loaded
        // while one is multiplied); beside resident blocks once
        constexpr int R = team_resident<M, B, NR, J>();
        constexpr int N = R > 0 ? 2 : (std::is_same<M, Dict>::value ? 8 : (B * NR == 2 ? 4 : 2));
        typedef TeamGroup<M, B, N> Group;
        TeamRes<M, B, R> res[J];
        Group cur;
        {
            TeamPtr A = team_args();
#pragma unroll
            for (int j = 0; j < J; j++) {
                const Slice sl = slice_of(j);
                res[j].load(A->t.lidx, A->a.vw, A->a.nslots, sl.s0, sl.width, lane);
            }
            if (R == 0) {
                const Slice sl = first_slice;
                cur.load(A->t.lidx, A->a.vw, A->a.nslots, sl.s0, sl.width, lane);
            }
        }
        // What the quick iterations know of the problem's record; lane k of
        // each wavefront has right-hand side k.
        int dmask;
        int64_t iters, due;
        double rr_need, rho_keep = 0.;
        bool pending, refined = true;   // refined: the latest residual sums are a refinement's
        auto quick_state = [&] {
            const int k = lane < NR ? lane : NR - 1;
            dmask = 0;
            for (int i = 0; i < NR; i++) dmask |= (P.done[i] ? 1 : 0) << i;
            iters = P.iters;
            due = P.maxit - P.last_ckpt < P.ckpt_interval ? P.maxit : P.last_ckpt + P.ckpt_interval;
            // rr < drop, or rr <= target
            const double drop = P.drop * P.drop * P.rr_ckpt[k];
            const double below = drop > 0. ? __longlong_as_double(__double_as_longlong(drop) - 1) : -1.;
            rr_need = fmax(below, P.rr_target[k]);
            pending = P.ckpt_pending != 0;
        };
        __syncthreads();
        quick_state();
        int period = 0;
        const int ce = A0->t.ce, max_periods = A0->t.max_periods;
        while (!s_bad && period < max_periods) {
            bool running = true;
            for (int it = 0; it < ce && running; it++) {
                // ---- K1: q = Ks p, sums of p.q, q.z, q.Mq
                fresh();
                qs++;
                TeamPtr A = team_args();
                const uint16_t *lidx = A->t.lidx;
                const void *vw_ = A->a.vw, *minv = A->a.minv;
                const int64_t ns = A->a.nslots;
                Slice sls[J];
#pragma unroll
                for (int j = 0; j < J; j++) sls[j] = slice_of(j);
#pragma unroll
                for (int j = 0; j < J; j++) {
                    const Slice &sl = sls[j], &after = sls[(j + 1) % J];
                    double acc[NR][B];
#pragma unroll
                    for (int k = 0; k < NR; k++)
#pragma unroll
                        for (int i = 0; i < B; i++) acc[k][i] = 0.;
                    auto block = [&](uint32_t li, const TeamBlk<M, B> &blk) {
                        W tv[NR][B];
                        rec_load<W, B, NR>(lp + REC * li, tv);
#pragma unroll
                        for (int jj = 0; jj < B; jj++)
#pragma unroll
                            for (int i = 0; i < B; i++) {
                                const double m = blk.at(tab, jj * B + i);
#pragma unroll
                                for (int k = 0; k < NR; k++) acc[k][i] = mac(m, (double)tv[k][jj], acc[k][i]);
                            }
                    };
                    int kb = 0;
                    if constexpr (R > 0) {
                        if (R < sl.width) cur.load(lidx, vw_, ns, sl.s0 + R * WAVE, sl.width - R, lane);
#pragma unroll
                        for (; kb < R; kb += 4)
                            if (kb < sl.width) {
                                res[j].keep(kb);
#pragma unroll
                                for (int u = 0; u < 4; u++) block(res[j].col(kb + u), res[j].blk[kb + u]);
                            }
                        while (kb < sl.width) {
#pragma unroll
                            for (int u = 0; u < N; u++) block(cur.li[u], cur.blk[u]);
                            kb += N;
                            if (kb < sl.width) cur.load(lidx, vw_, ns, sl.s0 + (int64_t)kb * WAVE, sl.width - kb, lane);
                        }
                    } else {
                        // one group at least (an absent slice's is null), and
                        // while it is multiplied the next one's loads: of this
                        // slice, of the next, or of the first in the next
                        // iteration (its wait is then the exchange's)
                        do {
                            Group next;
                            kb += N;
                            const bool more = kb < sl.width;
                            next.load(lidx, vw_, ns, more ? sl.s0 + (int64_t)kb * WAVE : after.s0,
                                      more ? sl.width - kb : after.width, lane);
#pragma unroll
                            for (int u = 0; u < N; u++) block(cur.li[u], cur.blk[u]);
                            cur = next;
                        } while (kb < sl.width);
                    }
                    double v[3 * NR];
#pragma unroll
                    for (int i = 0; i < 3 * NR; i++) v[i] = 0.;
                    if (sl.own) {
                        W mi[B * B];
                        team_minv<W, B, BJ>(minv, sl.row, mi);
                        W po[NR][B];
                        rec_load<W, B, NR>(lp + REC * ((wave + j * TEAM_WAVES) * WAVE + lane), po);
#pragma unroll
                        for (int k = 0; k < NR; k++) {
                            W zv[B], mq[B];
#pragma unroll
                            for (int i = 0; i < B; i++) q[j][k][i] = (W)acc[k][i];
                            precond<W, B, BJ>(mi, r[j][k], zv);
                            precond<W, B, BJ>(mi, q[j][k], mq);
#pragma unroll
                            for (int i = 0; i < B; i++) {
                                v[k] = mac((double)po[k][i], (double)q[j][k][i], v[k]);
                                v[NR + k] = mac((double)q[j][k][i], (double)zv[i], v[NR + k]);
                                v[2 * NR + k] = mac((double)q[j][k][i], (double)mq[i], v[2 * NR + k]);
                            }
                        }
                        export_row(j, sl.row, q[j], qs);
                    }
                    slice_sums(v, std::integral_constant<int, 3 * NR>(), 0, j);
                }
                __syncthreads();
                xs++;
                publish(0, 3 * NR, xs);
                // ---- R: the same scalars in every member
                fresh();
                double al64[NR];
                W be[NR];
                bool slot = false;
                const bool ck = refined;
                refined = false;
                collect(ck ? NVC : NVN, xs, G > 1 ? qs : 0);
                // Most iterations need alpha and beta, which every wavefront forms for itself, and whether a
                // refinement is due or something went wrong (reduce_rhs and
                // reduce_finish without their records: those cost 1800
                // cycles on the way from the sums to the update, this 500).
                // (With more slices a wavefront the registers for a period's last
                // iteration are not there.)
                bool quick = !ck && (J == 1 || it != ce - 1);
                if (quick) {
                    const int k = lane < NR ? lane : NR - 1;
                    auto sum_of = [&](int v) { return NR == 1 && G == 1 ? lane_value(own_total, v) : red[v + k]; };
                    const double pq = sum_of(0), qz = sum_of(NR), qmq = sum_of(2 * NR), rho = sum_of(3 * NR),
                                 rr = sum_of(3 * NR + NRES - NR);
                    const bool dn = dmask >> k & 1;
                    const double alpha = dn ? 0. : (pq != 0. ? rho / pq : 0.);
                    const double rho1 = mac(alpha * alpha, qmq, mac(-2. * alpha, qz, rho));
                    const double beta = dn ? 0. : (rho != 0. ? rho1 / rho : 0.);
                    quick = !__any(!dn && (!(pq == pq) || !(rho == rho) || !(qz == qz) || !(qmq == qmq)));
                    bool due_now = false;
                    if constexpr (J == 1) {
                        due_now = pending || __any(!dn && rr <= rr_need) || iters + 1 >= due;
                        quick = quick && !(due_now && it == ce - 1);   // the refinement's slot
                    }
                    if (quick) {
                        if constexpr (J == 1) rho_keep = rho1;
                        else if (wave == 0 && lane < NR && !dn) P.rho_pred[k] = rho1;   // for the next refinement's
                        iters++;
                        if constexpr (J == 1) pending = due_now;
                        else if (__any(!dn && rr <= rr_need) || iters >= due) pending = true;
#pragma unroll
                        for (int kk = 0; kk < NR; kk++) {
                            al64[kk] = NR == 1 ? alpha : lane_value(alpha, kk);
                            be[kk] = (W)(NR == 1 ? beta : lane_value(beta, kk));
                        }
                    }
                }
                if (!quick) {
                    if (wave == 0) {
                        int f = 0;
                        if (J == 1 && lane < NR && iters != P.iters && !P.done[lane]) P.rho_pred[lane] = rho_keep;
                        if (lane == 0) {
                            P.iters = iters;
                            if (pending) P.ckpt_pending = 1;
                        }
                        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        if (lane < NR) {
                            const int k = lane;
                            f = reduce_rhs(P, k, red[k], red[NR + k], red[2 * NR + k], red[3 * NR + k],
                                           red[3 * NR + NRES - NR + k], ck ? red[NVN + k] : 0., ck ? red[NVN + NR + k] : 0.,
                                           ck);
                        }
                        for (int k = 1; k < NR; k++) f |= __shfl(f, k, WAVE);
                        if (lane == 0) {
                            reduce_finish(P, f, ck);
                            // a refinement comes: whether any workgroup gave up
                            if (G > 1 && it == ce - 1 && P.ckpt_pending &&
                                __hip_atomic_load(team_args_of<false>()->t.ctl + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                                s_bad = 1;
                        }
                    }
                    __syncthreads();
                    if (s_bad) break;
                    running = P.status == ST_RUNNING;
                    if (!running) break;
                    slot = it == ce - 1 && P.ckpt_pending;
                    quick_state();
#pragma unroll
                    for (int k = 0; k < NR; k++) {
                        al64[k] = P.alpha[k];
                        be[k] = (W)P.beta[k];
                    }
                }
                fresh();
                // ---- K2: y, r, p of the own rows and of the halo.  A
                // finished right-hand side has alpha = beta = 0: its y and r
                // stay as they are, and its p feeds nothing any more.
                W al[NR];
#pragma unroll
                for (int k = 0; k < NR; k++) al[k] = (W)al64[k];
                rp ^= 1;
                auto k2_row = [&](W(*pk)[B], W(*rk)[B], const W(*qk)[B], const W *mi, auto each) {
#pragma unroll
                    for (int k = 0; k < NR; k++) {
                        W zv[B];
#pragma unroll
                        for (int i = 0; i < B; i++) rk[k][i] = mac(-al[k], qk[k][i], rk[k][i]);
                        precond<W, B, BJ>(mi, rk[k], zv);
#pragma unroll
                        for (int i = 0; i < B; i++) {
                            pk[k][i] = mac(be[k], pk[k][i], zv[i]);
                            each(k, rk[k][i], zv[i]);
                        }
                    }
                };
                minv = team_args()->a.minv;
#pragma unroll
                for (int j = 0; j < J; j++) {
                    const Slice sl = slice_of(j);
                    double v[NRES];
#pragma unroll
                    for (int i = 0; i < NRES; i++) v[i] = 0.;
                    if (sl.own) {
                        W *pl = lp + REC * ((wave + j * TEAM_WAVES) * WAVE + lane);
                        W po[NR][B];
                        rec_load<W, B, NR>(pl, po);
#pragma unroll
                        for (int k = 0; k < NR; k++)
#pragma unroll
                            for (int i = 0; i < B; i++) y[j][k][i] = mac(al64[k], (double)po[k][i], y[j][k][i]);
                        if (!slot) {
                            W mi[B * B];
                            team_minv<W, B, BJ>(minv, sl.row, mi);
                            k2_row(po, r[j], q[j], mi, [&](int k, W rv, W zv) {
                                v[k] = mac((double)rv, (double)zv, v[k]);
                                if constexpr (BJ) v[NR + k] = mac((double)rv, (double)rv, v[NR + k]);
                            });
                            rec_store<W, B, NR>(pl, po);
                        }
                    }
                    if (!slot) slice_sums(v, std::integral_constant<int, NRES>(), 3 * NR, j);
                }
                if (!slot)
                    import_rows(qs, std::true_type(), [&](int h, int gr, W(*qv)[B]) {
                        W mi[B * B];
                        team_minv<W, B, BJ>(minv, gr, mi);
                        W *pl = lp + REC * (rows + h), *rl = lr + REC * h;
                        W po[NR][B], ro[NR][B];
                        rec_load<W, B, NR>(pl, po);
                        rec_load<W, B, NR>(rl, ro);
                        k2_row(po, ro, qv, mi, [](int, W, W) {});
                        rec_store<W, B, NR>(pl, po);
                        rec_store<W, B, NR>(rl, ro);
                    });
                __syncthreads();
                if (!slot) publish(3 * NR, NVN, xs + 1);
                else if (tid == 0) P.src_ckpt = 1;
                if (it == ce - 1 && s_bad) break;   // (a wait that gave up: the quick iterations do not look)
            }
            if (!running || s_bad) break;
            period++;
            if (mb.m == 0 && tid == 0)
                __hip_atomic_fetch_add(team_args()->t.ctl + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (P.ckpt_pending) {
                refine(false);
                refined = true;
            }
        }
        seq_max = seq_max > xs ? seq_max : xs;
        seq_max = seq_max > qs ? seq_max : qs;
        if (J == 1 && tid == 0 && !s_bad) P.iters = iters;
        __syncthreads();
        if (mb.m == 0 && !s_bad)
            for (int i = tid; i < (int)(sizeof(ProbDev) / 4); i += TEAM_WG)
                reinterpret_cast<uint32_t *>(gP)[i] = reinterpret_cast<const uint32_t *>(&P)[i];
    }
    if (tid == 0) atomicMax(team_args()->t.ctl + 3, seq_max);
}

typedef void (*TeamFn)(TeamAll);

// Slices a wavefront can hold in its registers: each takes NR B (8 + 2
// sizeof(W)) bytes of y, r and q a lane, up to 96 of its 256 registers; the
// product's blocks in flight and the sums take the rest.
template <typename W, int B, int NR> constexpr int team_jmax()
{
    constexpr int regs = NR * B * (8 + 2 * (int)sizeof(W)) / 4;
    return regs * 8 <= 96 ? 8 : (regs * 4 <= 96 ? 4 : (regs * 2 <= 96 ? 2 : 1));
}
template <typename W, typename M, int B, int NR, bool BJ> TeamFn team_j(int j)
{
    constexpr int JM = team_jmax<W, B, NR>();
    if (j <= 1) return k_cg_team<W, M, B, NR, BJ, 1>;
    if constexpr (JM >= 2)
        if (j <= 2) return k_cg_team<W, M, B, NR, BJ, 2>;
    if constexpr (JM >= 4)
        if (j <= 4) return k_cg_team<W, M, B, NR, BJ, 4>;
    if constexpr (JM >= 8)
        if (j <= 8) return k_cg_team<W, M, B, NR, BJ, 8>;
    return nullptr;
}
template <typename W, typename M> TeamFn team_pick(int b, int nr, bool bj, int j)
{
    if (b == 2) {
        if (nr == 1) return bj ? team_j<W, M, 2, 1, true>(j) : team_j<W, M, 2, 1, false>(j);
        return bj ? team_j<W, M, 2, 3, true>(j) : team_j<W, M, 2, 3, false>(j);
    }
    if (nr == 1) return bj ? team_j<W, M, 3, 1, true>(j) : team_j<W, M, 3, 1, false>(j);
    return bj ? team_j<W, M, 3, 3, true>(j) : team_j<W, M, 3, 3, false>(j);
}
// The kernels, one translation unit per matrix format; nullptr: more slices
// per wavefront than the registers hold.
TeamFn team_fn_fp64(int b, int nr, bool bj, int j);
TeamFn team_fn_fix48(int b, int nr, bool bj, int j);
TeamFn team_fn_dict(int b, int nr, bool bj, int j);

} // namespace amie
