// Host side of the team CG (team.hpp): how a batch's problems are cut into
// members, the halo plan, and the launch.
#include <algorithm>
#include <cmath>
#include <functional>
#include <queue>

#include "batch.hpp"
#include "team.hpp"

namespace amie {

// One workgroup per member: the rows of other members that its blocks name
// (padding blocks left out), as a bitmap of the problem's rows in LDS.
// loc: per slice {member's local slice, member of its problem} packed.
// fill = 0 counts them; fill = 1 writes the list (rows in order), the slots'
// local columns and the marks of the exported rows.
__global__ __launch_bounds__(TEAM_WG) void k_team_halo(SolveArgs a, const TeamMember *members, const int32_t *mslice,
                                                      const uint32_t *loc, const int32_t *row_len, int fill,
                                                      int32_t *count, uint32_t *halo, uint16_t *lidx, uint8_t *exported)
{
    extern __shared__ uint32_t bits[];
    __shared__ int32_t start[TEAM_WG + 1];
    const TeamMember mb = members[blockIdx.x];
    const int tid = threadIdx.x, wave = wave_id(), lane = tid % WAVE;
    // the problem's slices
    const int last = mb.tile0 + mb.ntiles - 1;
    const int64_t prow0 = (int64_t)a.tile_slice0[mb.tile0] * WAVE;
    const int64_t nrows = (int64_t)(a.tile_slice0[last] + a.tile_nslices[last]) * WAVE - prow0;
    const int nw = (int)((nrows + 31) / 32), per = (nw + TEAM_WG - 1) / TEAM_WG;
    for (int i = tid; i < nw; i += TEAM_WG) bits[i] = 0;
    __syncthreads();
    auto slots = [&](auto use) {
        for (int s = wave; s < mb.nsl; s += TEAM_WAVES) {
            const int gl = mslice[mb.sl0 + s];
            if (gl < 0) continue;
            const int4 sd = a.slice_desc[gl];
            const int64_t sp = ((int64_t)(uint32_t)sd.x | ((int64_t)sd.y << 32)) + lane;
            const int len = lane < sd.w ? row_len[(int64_t)gl * WAVE + lane] : 0;
            for (int k = 0; k < sd.z; k++) {
                const int64_t slot = sp + (int64_t)k * WAVE;
                use(s, slot, k < len ? (int)a.col[slot] : -1);
            }
        }
    };
    slots([&](int, int64_t, int c) {
        if (c >= 0 && loc[c / WAVE] >> 16 != (uint32_t)mb.m) atomicOr(&bits[(c - prow0) >> 5], 1u << ((c - prow0) & 31));
    });
    __syncthreads();
    // rows marked before each thread's run of words
    const int w0 = min(nw, tid * per), w1 = min(nw, w0 + per);
    int n = 0;
    for (int i = w0; i < w1; i++) n += __popc(bits[i]);
    start[tid + 1] = n;
    if (tid == 0) start[0] = 0;
    __syncthreads();
    if (tid == 0)
        for (int i = 0; i < TEAM_WG; i++) start[i + 1] += start[i];
    __syncthreads();
    if (!fill) {
        if (tid == 0) count[blockIdx.x] = start[TEAM_WG];
        return;
    }
    n = start[tid];
    for (int i = w0; i < w1; i++)
        for (uint32_t b = bits[i]; b; b &= b - 1) {
            const uint32_t row = (uint32_t)(prow0 + (int64_t)i * 32 + __builtin_ctz(b));
            halo[mb.halo0 + n++] = row;
            exported[row] = 1;   // every writer stores the same value
        }
    slots([&](int s, int64_t slot, int c) {
        int li = s * WAVE + lane;   // a padding block (zero) reads its own row
        if (c >= 0) {
            const uint32_t l = loc[c / WAVE];
            if (l >> 16 == (uint32_t)mb.m) {
                li = (int)(l & 0xffffu) * WAVE + c % WAVE;
            } else {
                const int word = (int)((c - prow0) >> 5), t = word / per;
                li = mb.nsl * WAVE + start[t];
                for (int i = t * per; i < word; i++) li += __popc(bits[i]);
                li += __popc(bits[word] & ((1u << ((c - prow0) & 31)) - 1u));
            }
        }
        lidx[slot] = (uint16_t)li;
    });
}

namespace {

constexpr size_t LDS_BYTES = 160 * 1024;
// The largest dynamic LDS of a kernel is a property of the function, not of a
// launch: always set to the same, so that batches on other threads (a server
// builds several at a time) never lower it between here and a launch.
constexpr size_t HALO_LDS = LDS_BYTES - 8192;   // the bitmap beside k_team_halo's counts

template <typename W> int team_jmax_of(int b, int nr)
{
    if (b == 2) return nr == 1 ? team_jmax<W, 2, 1>() : team_jmax<W, 2, 3>();
    return nr == 1 ? team_jmax<W, 3, 1>() : team_jmax<W, 3, 3>();
}

// Tiles per member.  A small problem is spread until a member reads about
// 160 KB of matrix an iteration (1 us at the 64 bytes a clock that a CU gets
// from L2, what an exchange costs); one of at most four tiles stays with one
// member, which exchanges nothing.  A larger batch takes as many members as
// there are CUs, then the most tiles that the registers hold.  0: a problem
// does not fit a team of every CU.
int team_tiles(const Batch &B, int jmax, double slot_bytes)
{
    const int cus = std::max(1, B.ctx->num_cu), most = TEAM_WAVES * jmax / TILE_SLICES;
    const double tile_bytes = slot_bytes * (double)B.nslots / std::max<double>(1., (double)B.ntiles);
    int tpw = std::max(1, std::min(4, (int)(160e3 / tile_bytes)));
    int big = 0;
    for (const ProbHost &P : B.ph) big = std::max(big, P.ntiles);
    tpw = big <= 4 ? big : tpw;
    tpw = std::min(tpw, most);
    if (B.team_tiles > 0) {
        tpw = std::min(B.team_tiles, most);
        return (big + tpw - 1) / tpw > cus ? 0 : tpw;
    }
    auto members = [&](int t) {
        int64_t n = 0;
        for (const ProbHost &P : B.ph) n += (P.ntiles + t - 1) / t;
        return n;
    };
    while (tpw < most && members(tpw) > cus) tpw++;
    return (big + tpw - 1) / tpw > cus ? 0 : tpw;
}

// The choice between the two paths, which give the same bits: estimated times
// of a solve by each, in microseconds an iteration of a problem with a weight
// of one.  Both follow what was measured (an MI355X, 205 batches of one to 64
// problems by element, precision and right-hand sides, team and launches in
// turn; the estimates' spread is about 10 %):
//   launches   a floor of three dependent kernels and the stream of the matrix
//              and the vectors at 4-6 TB/s, with a share a block for the
//              value-indexed matrix.  They overlap where rows are long (3 x 3
//              blocks) and add up where they are short.  A problem that is
//              done leaves the iteration.
//   team       a fixed part (sums, exchange, scalars), the product of the
//              tiles a member holds, and the halo words of all members that
//              run at a time, which come past the caches at 0.6-1 TB/s.
//              Members are claimed in order, and a team whose last member has
//              to wait for a CU keeps the others idle.
// Almost everywhere the team is the faster one (1.1 to 6 times).  It is not
// where teams of more than half the chip come one after the other (three
// loads in FP64, a workgroup holds four tiles: 20 RVEs of 87..512 cells 357 us
// an iteration against 277, two of 512 cells 95 against 88; but 64 of 36..256
// cells 159 against 220) and where 3 x 3 blocks by value index read the table
// for many slices in turn (12 RVEs of 19..48 cells: 101 against 76).
struct Pace {
    double fixed, tile[3];   // a tile with at most 2, 4 and 8 slices a wavefront
};
constexpr Pace PACE[3][2][2] = {   // FP64, FIX48 planes, value-indexed; 2 x 2, 3 x 3; one and three right-hand sides
    {{{3.2, {0.3, 1.6, 1.6}}, {2.6, {1.9, 1.9, 1.9}}}, {{6.3, {0.3, 6.1, 6.1}}, {8.2, {5.2, 5.2, 5.2}}}},
    {{{4.4, {0.3, 1.4, 1.4}}, {2.0, {1.8, 1.8, 1.8}}}, {{4.7, {2.2, 3.2, 6.1}}, {7.7, {4.5, 4.5, 4.5}}}},
    {{{2.0, {0.7, 0.6, 0.7}}, {6.1, {0.3, 0.4, 0.4}}}, {{12.0, {0.4, 2.0, 5.3}}, {8.2, {4.8, 4.8, 4.8}}}},
};
// us a MB of halo words; a team of more than half the chip takes all of its
// words at the same time, nothing between them
constexpr double HALO_US_MB[2][2] = {{1.0, 1.25}, {1.75, 0.9}}, HALO_ALONE = 1.15;
struct Launches {
    double floor, tbs, block;   // us; TB/s; us per 10^6 value-indexed blocks
};
constexpr Launches LAUNCHES[2][2] = {{{16., 5.9, 1.8}, {23., 5.6, 2.9}}, {{24., 5.0, 6.0}, {32., 4.1, 8.6}}};

// iterations of a problem, up to a factor: its nodes along one side
double weight_of(const Batch &B, const ProbHost &P) { return std::pow((double)P.nrows, 1. / B.et.b); }

double launch_estimate(const Batch &B, const std::vector<int32_t> &probs, bool f64, bool indexed)
{
    const int b = B.et.b, w = f64 ? 8 : 4;
    const Launches &L = LAUNCHES[b - 2][B.nrhs > 1];
    const double blocks = (double)B.nslots / std::max<double>(1., (double)B.nrows_pad) * WAVE * TILE_SLICES;   // a tile's
    const double bytes = blocks * (indexed ? 4. : (f64 ? 8. : 6.) * b * b + 4.) +
                         WAVE * TILE_SLICES * b * B.nrhs * (8.75 * w + 4.);
    const double tile = bytes / L.tbs * 1e-6 + (indexed ? L.block * blocks * 1e-6 : 0.);
    std::vector<std::pair<double, int>> by;   // the shortest solves end first
    double active = 0., t = 0., done = 0.;
    for (int p : probs) {
        by.push_back({weight_of(B, B.ph[p]), B.ph[p].ntiles});
        active += B.ph[p].ntiles;
    }
    std::sort(by.begin(), by.end());
    for (auto &e : by) {
        const double s = tile * active;
        t += (e.first - done) * (b == 2 ? L.floor + s : std::hypot(L.floor, s));
        done = e.first;
        active -= e.second;
    }
    return t;
}

double team_estimate(const Batch &B, const TeamPlan &T, const std::vector<int32_t> &probs, bool f64, bool indexed, int j)
{
    const int b = B.et.b, nr = B.nrhs, cus = std::max(1, B.ctx->num_cu);
    const Pace &C = PACE[f64 ? 0 : (indexed ? 2 : 1)][b - 2][nr > 1];
    const double tile = C.tile[j <= 2 ? 0 : (j <= 4 ? 1 : 2)];
    int64_t members = 0, halos = 0;
    for (int p : probs) {
        members += T.first[p + 1] - T.first[p];
        for (int m = T.first[p]; m < T.first[p + 1]; m++) halos += T.nhalo[m];
    }
    const double us = HALO_US_MB[b - 2][nr > 1] * 8e-6 * b * nr * (f64 ? 2 : 1) * (double)std::min<int64_t>(members, cus);
    const double mean = (double)halos / (double)std::max<int64_t>(1, members);
    std::priority_queue<double, std::vector<double>, std::greater<double>> cu;   // when each is free
    for (int i = 0; i < cus; i++) cu.push(0.);
    double end = 0.;
    for (int p : probs) {
        const int G = T.first[p + 1] - T.first[p];
        double halo = 0., from = 0.;
        for (int m = T.first[p]; m < T.first[p + 1]; m++) halo += T.nhalo[m];
        for (int m = 0; m < G; m++) {
            from = std::max(from, cu.top());
            cu.pop();
        }
        halo /= std::max(1, G);
        if (b == 3) halo = 0.5 * (halo + mean);   // (other problems' halos are smaller)
        const double to = from + weight_of(B, B.ph[p]) * (C.fixed + tile * std::min(T.tpw, B.ph[p].ntiles) +
                                                          (2 * G > cus ? HALO_ALONE : 1.) * us * halo);
        for (int m = 0; m < G; m++) cu.push(to);
        end = std::max(end, to);
    }
    return end;
}

} // namespace

// The plan of a batch for `tpw` tiles per member, made once per batch.  A
// member's tiles are neighbours in the original numbering (rows sorted by
// length inside windows put a tile's own neighbours in other tiles, and a
// run of the sorted order would have most of its window as halo).
static int team_plan(Batch &B, int tpw, TeamPlan **out)
{
    *out = nullptr;
    for (auto &p : B.team_plans)
        if (p->tpw == tpw) {
            *out = p.get();
            return AMIE_OK;
        }
    // without memory for a plan the launch path runs, which needs none
    auto no_room = [] {
        (void)hipGetLastError();
        return AMIE_OK;
    };
    std::unique_ptr<TeamPlan> T(new TeamPlan());
    T->tpw = tpw;
    std::vector<TeamMember> mem;
    std::vector<int32_t> mslice, mtile;
    std::vector<uint32_t> loc((size_t)B.nslices, 0);
    int64_t xb = 0, rows_max = 0;
    T->first.resize(B.nprob + 1);
    T->ok = true;
    for (int p = 0; p < B.nprob; p++) {
        const ProbHost &P = B.ph[p];
        T->first[p] = (int32_t)mem.size();
        std::vector<int64_t> sum((size_t)P.ntiles, 0);
        std::vector<int32_t> cnt((size_t)P.ntiles, 0), order((size_t)P.ntiles);
        constexpr int TR = TILE_SLICES * WAVE;
        for (int64_t o = 0; o < P.nrows; o++) {
            sum[P.iperm[o] / TR] += o;
            cnt[P.iperm[o] / TR]++;
        }
        for (int t = 0; t < P.ntiles; t++) order[t] = t;
        const int G = (P.ntiles + tpw - 1) / tpw;
        if (G > 1)   // (a member of its own keeps the tiles' order: it sums them from LDS)
            std::stable_sort(order.begin(), order.end(),
                             [&](int x, int y) { return sum[x] / std::max(1, cnt[x]) < sum[y] / std::max(1, cnt[y]); });
        for (int m = 0; m < G; m++) {
            TeamMember t{};
            t.prob = p;
            t.m = m;
            t.G = G;
            t.sl0 = (int32_t)mslice.size();
            t.mt0 = (int32_t)mtile.size();
            t.tile0 = P.tile0;
            t.ntiles = P.ntiles;
            t.xb = xb;
            for (int i = m * tpw; i < std::min(P.ntiles, (m + 1) * tpw); i++) {
                mtile.push_back(order[i]);
                for (int u = 0; u < TILE_SLICES; u++) {
                    const int s = order[i] * TILE_SLICES + u;
                    if (s < P.nslices) loc[P.slice0 + s] = (uint32_t)m << 16 | (uint32_t)(mslice.size() - t.sl0);
                    mslice.push_back(s < P.nslices ? P.slice0 + s : -1);
                }
            }
            t.nsl = (int32_t)mslice.size() - t.sl0;
            mem.push_back(t);
        }
        // tile values and sums of two exchanges
        xb += 2ll * 7 * B.nrhs * (P.ntiles + 1);
        rows_max = std::max(rows_max, (int64_t)P.nslices * WAVE);
        if (2ll * 7 * B.nrhs * (P.ntiles + 1) > (1 << 28)) T->ok = false;   // 32-bit indices of the values
    }
    T->first[B.nprob] = (int32_t)mem.size();
    const size_t bitmap = (size_t)((rows_max + 31) / 32) * 4;
    if (bitmap > HALO_LDS || mslice.size() >= INT32_MAX || B.max_width > 65535) T->ok = false;
    if (T->ok) {
        const int nm = (int)mem.size();
        const hipStream_t st = B.stream;
        if (!T->members.alloc(nm * sizeof(TeamMember)) || !T->mslice.alloc(mslice.size() * 4) ||
            !T->mtile.alloc(mtile.size() * 4) || !T->loc.alloc(loc.size() * 4) || !T->count.alloc((size_t)nm * 4) ||
            !T->lidx.alloc((size_t)B.nslots * 2) || !T->exported.alloc((size_t)B.nrows_pad) ||
            !T->xb.alloc((size_t)xb * 16) || !T->order.alloc((size_t)nm * 4))
            return no_room();
        AMIE_HIP(hipFuncSetAttribute((const void *)k_team_halo, hipFuncAttributeMaxDynamicSharedMemorySize, (int)HALO_LDS));
        AMIE_HIP(hipMemcpyAsync(T->members.p, mem.data(), nm * sizeof(TeamMember), hipMemcpyHostToDevice, st));
        AMIE_HIP(hipMemcpyAsync(T->mslice.p, mslice.data(), mslice.size() * 4, hipMemcpyHostToDevice, st));
        AMIE_HIP(hipMemcpyAsync(T->mtile.p, mtile.data(), mtile.size() * 4, hipMemcpyHostToDevice, st));
        AMIE_HIP(hipMemcpyAsync(T->loc.p, loc.data(), loc.size() * 4, hipMemcpyHostToDevice, st));
        AMIE_HIP(hipMemsetAsync(T->exported.p, 0, T->exported.n, st));
        AMIE_HIP(hipMemsetAsync(T->xb.p, 0, T->xb.n, st));
        AMIE_HIP(hipMemsetAsync(T->lidx.p, 0, T->lidx.n, st));   // the null slots read row 0
        const SolveArgs a = B.args(AMIE_FP64);
        auto halo = [&](int fill) {
            hipLaunchKernelGGL(k_team_halo, dim3(nm), dim3(TEAM_WG), bitmap, st, a, T->members.as<TeamMember>(),
                               T->mslice.as<int32_t>(), T->loc.as<uint32_t>(), B.row_len.as<int32_t>(), fill,
                               T->count.as<int32_t>(), T->halo.as<uint32_t>(), T->lidx.as<uint16_t>(),
                               T->exported.as<uint8_t>());
        };
        halo(0);
        AMIE_HIP(hipGetLastError());
        std::vector<int32_t> h(nm);
        AMIE_HIP(hipMemcpyAsync(h.data(), T->count.p, (size_t)nm * 4, hipMemcpyDeviceToHost, st));
        AMIE_HIP(hipStreamSynchronize(st));
        int64_t total = 0;
        for (int i = 0; i < nm; i++) {
            mem[i].halo0 = (int32_t)total;
            mem[i].nhalo = h[i];
            total += h[i];
            const int64_t rows = (int64_t)mem[i].nsl * WAVE;
            T->lds_units = std::max<int64_t>(T->lds_units, rows + 2 * (int64_t)h[i]);
            if (rows + h[i] > 65536) T->ok = false;   // 16-bit local columns
        }
        T->nhalo.swap(h);
        if (total >= INT32_MAX) T->ok = false;
        if (T->ok) {
            if (!T->halo.alloc((size_t)total * 4)) return no_room();
            AMIE_HIP(hipMemcpyAsync(T->members.p, mem.data(), nm * sizeof(TeamMember), hipMemcpyHostToDevice, st));
            halo(1);
            AMIE_HIP(hipGetLastError());
            AMIE_HIP(hipStreamSynchronize(st));
        }
    }
    B.team_plans.push_back(std::move(T));
    *out = B.team_plans.back().get();
    return AMIE_OK;
}

// Whether (and how) a pass over the problems in `subset` runs as a team
// launch: R.team is set when it does.  The other paths take what does not
// fit: precisions without a team kernel, problems of more rows than the chip
// holds, halos that outgrow the LDS.
int team_prepare(Batch &B, SolveRun &R, const std::vector<char> &subset)
{
    R.team = nullptr;
    const int mode = R.mode;
    if ((mode != AMIE_FP64 && mode != AMIE_MIXED_FIX48) || R.o.time_kernels || R.o.persistent > 0 || R.o.use_graph ||
        B.team_use == AMIE_TEAM_NEVER || B.team_gave_up)
        return AMIE_OK;
    const bool f64 = mode == AMIE_FP64;
    const int b = B.et.b, nr = B.nrhs, w = f64 ? 8 : 4;
    const int jmax = f64 ? team_jmax_of<double>(b, nr) : team_jmax_of<float>(b, nr);
    // the value-indexed matrix where its table fits beside p, else the planes
    // (the same values)
    const bool indexed = !f64 && B.k1_format(mode, R.bj) == 1;
    const int tpw = team_tiles(B, jmax, 2. + (indexed ? 2. : (f64 ? 8. : 6.) * b * b));
    if (!tpw) return AMIE_OK;
    TeamPlan *T = nullptr;
    if (int rc = team_plan(B, tpw, &T)) return rc;
    if (!T || !T->ok) return AMIE_OK;
    const int j = (tpw * TILE_SLICES + TEAM_WAVES - 1) / TEAM_WAVES;
    const size_t vec = team_lds(T->lds_units, b, nr, w);
    const size_t table = indexed ? (size_t)B.dict_n * (b == 2 ? DictEntry<2>::N : DictEntry<3>::N) * 8 : 0;
    auto fits = [&](TeamFn fn, size_t dyn) -> bool {
        hipFuncAttributes fa{};
        if (hipFuncGetAttributes(&fa, (const void *)fn) != hipSuccess) return false;
        R.team_lds_most = LDS_BYTES - fa.sharedSizeBytes;
        return fa.sharedSizeBytes + dyn <= LDS_BYTES;
    };
    TeamFn fn = nullptr;
    size_t dyn = vec;
    if (indexed) {
        fn = team_fn_dict(b, nr, R.bj, j);
        dyn = table + vec;
        R.a.vw = B.dict_ids.p;
        if (!fn || !fits(fn, dyn)) fn = nullptr;
    }
    if (!fn) {
        dyn = vec;
        R.a.vw = f64 ? B.vs64.p : B.vfx.p;
        fn = f64 ? team_fn_fp64(b, nr, R.bj, j) : team_fn_fix48(b, nr, R.bj, j);
        if (!fn || !fits(fn, dyn)) {
            if (indexed) R.a.vw = B.dict_ids.p;   // as apply_tuned left it
            return AMIE_OK;
        }
    }
    // members in the order they are claimed: the largest problems first, the
    // members of a problem in a row
    std::vector<int32_t> probs, order;
    for (int p = 0; p < B.nprob; p++)
        if (subset[p]) probs.push_back(p);
    std::stable_sort(probs.begin(), probs.end(), [&](int x, int y) { return B.ph[x].ntiles > B.ph[y].ntiles; });
    bool single = true;
    for (int p : probs) {
        for (int m = T->first[p]; m < T->first[p + 1]; m++) order.push_back(m);
        single = single && T->first[p + 1] - T->first[p] == 1;
    }
    if (B.team_use == AMIE_TEAM_AUTO) {
        const bool table = indexed && R.a.vw == B.dict_ids.p;
        const int key = (f64 ? 1 : 0) | (indexed ? 2 : 0) | (table ? 4 : 0);
        if (key != T->judged || probs != T->judged_probs) {
            T->pays = B.team_margin * team_estimate(B, *T, probs, f64, table, j) <= launch_estimate(B, probs, f64, indexed);
            T->judged = key;
            T->judged_probs = probs;
        }
        if (!T->pays) {
            if (indexed) R.a.vw = B.dict_ids.p;
            return AMIE_OK;
        }
    }
    if (order != T->h_order) {
        T->h_order.swap(order);   // kept: the source of the queued copy
        AMIE_HIP(hipMemcpyAsync(T->order.p, T->h_order.data(), T->h_order.size() * 4, hipMemcpyHostToDevice, B.stream));
    }
    R.team = T;
    R.team_fn = (const void *)fn;
    R.team_lds = dyn;
    R.team_single = single;
    R.team_first = probs.front();
    return AMIE_OK;
}

int team_plan_ahead(Batch &B, const amie_solve_opts &o)
{
    SolveRun R;
    R.o = o;
    R.mode = o.precision;
    R.bj = o.precond == AMIE_BLOCK_JACOBI;
    R.a = B.args(R.mode);
    if (int rc = team_prepare(B, R, std::vector<char>(B.nprob, 1))) return rc;
    AMIE_HIP(hipStreamSynchronize(B.stream));   // the copies to the device
    return AMIE_OK;
}

// Queues the pass's launch.
int team_launch(Batch &B, SolveRun &R)
{
    TeamPlan &T = *R.team;
    const hipStream_t s = B.stream;
    // the rows' words live in the buffers of the launch path's p sets (and y),
    // which hold no words of this path after a pass of that one
    if (B.team_dirty || B.team_seq > 0x7fffffffu) {
        for (DevBuf *v : {&B.p2, &B.p3, &B.p4, &B.y}) AMIE_HIP(hipMemsetAsync(v->p, 0, v->n, s));
        if (B.team_seq > 0x7fffffffu) {
            for (auto &t : B.team_plans)
                if (t->xb.p) AMIE_HIP(hipMemsetAsync(t->xb.p, 0, t->xb.n, s));
            B.team_seq = 0;
        }
        B.team_dirty = false;
    }
    AMIE_HIP(hipMemsetAsync(B.persist.p, 0, B.persist.n, s));
    TeamArgs ta{};
    ta.members = T.members.as<TeamMember>();
    ta.order = T.order.as<int32_t>();
    ta.nitems = (int32_t)T.h_order.size();
    ta.max_periods = (int32_t)std::min<int64_t>(INT32_MAX, std::max<int64_t>(0, R.max_periods));
    ta.ce = R.ce;
    ta.dict_n = (int32_t)B.dict_n;
    ta.mslice = T.mslice.as<int32_t>();
    ta.mtile = T.mtile.as<int32_t>();
    ta.lidx = T.lidx.as<uint16_t>();
    ta.halo = T.halo.as<uint32_t>();
    ta.exported = T.exported.as<uint8_t>();
    ta.xb = T.xb.as<uint64_t>();
    const bool f64 = R.mode == AMIE_FP64;
    // FP64 rows take a low and a high word: two buffers a parity
    ta.ql[0] = B.p2.as<uint64_t>();
    ta.qh[0] = B.p3.as<uint64_t>();
    ta.ql[1] = f64 ? B.p4.as<uint64_t>() : B.p3.as<uint64_t>();
    ta.qh[1] = B.y.as<uint64_t>();
    ta.seq0 = B.team_seq;
    ta.ctl = B.persist.as<uint32_t>();
    int grid = std::min(ta.nitems, std::max(1, B.ctx->num_cu));
    if (B.team_use == AMIE_TEAM_STARVED && !R.team_single) {
        // the largest problem's members come first: one workgroup too few for
        // them, and the error flag that a wait looks at is set
        const int p = R.team_first;
        grid = T.first[p + 1] - T.first[p] - 1;
        AMIE_HIP(hipMemsetAsync(B.persist.as<char>() + 8, 1, 1, s));
    }
    AMIE_HIP(hipFuncSetAttribute(R.team_fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)R.team_lds_most));
    TeamAll all{R.a, ta};
    void *kargs[] = {&all};
    // members of one team wait for each other: a cooperative launch, which
    // holds every workgroup resident; teams of one wait for nobody
    if (R.team_single)
        AMIE_HIP(hipLaunchKernel(R.team_fn, dim3(grid), dim3(TEAM_WG), kargs, R.team_lds, s));
    else
        AMIE_HIP(hipLaunchCooperativeKernel(R.team_fn, dim3(grid), dim3(TEAM_WG), kargs, (unsigned)R.team_lds, s));
    B.team_seq = UINT32_MAX;   // unknown (the next launch clears the words) until its end is seen
    AMIE_HIP(hipMemcpyAsync(B.h_persist_pinned, B.persist.p, 16, hipMemcpyDeviceToHost, s));
    return AMIE_OK;
}

} // namespace amie
