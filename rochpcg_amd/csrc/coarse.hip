// coarse.hip -- the V-cycle's coarsest levels in one workgroup.
//
// A level of a few thousand rows does not fill the GPU, and its sweeps are a
// chain of colours: as launches, 32 per level (15 on the coarsest), each about
// 2.7 us of launch and memory latency whatever it computes.  One workgroup
// orders its colours with a barrier instead and keeps every level's x, which
// the gathers read, in LDS, and the partial sums t too.  Values, columns and rhs
// come from L2 and do not depend on x: the workgroup's teams load the next
// steps' while one computes.
//
// What bounds a step is the instruction stream of one wave (a wave issues an
// instruction every four cycles): so the columns are laid out beforehand as LDS
// offsets, by section, with the unused slots of a group pointing at a zero
// behind the level's x.  A sum is then one LDS read and one multiply-add a
// slot, without masks or selects; the rest is a division and a barrier.  The value
// of an unused slot may be infinite, though it is no part of the sum: where any sum
// has come out as NaN, the V-cycle is run again over the used slots alone (CM_USED).
//
// Measured, a CG iteration of FP64 / mixed with every level as launches and with
// its coarse levels here: 16^3 253 / 238 -> 139 / 115 us, 32^3 279 / 257 ->
// 212 / 176 us, 64^3 380 / 315 -> 355 / 267 us, 104^3 562 / 421 -> 547 / 393 us;
// a step takes 0.5-0.9 us.
//
// Per row the arithmetic is that of the row_* functions of kernels.hpp, on the same
// stored values, slot by slot in the same order (an unused slot adds a * 0), so
// results are the same (but for the sign of a sum that is zero).
// The inner levels' r and x are left in the level vectors, as the launches leave
// them.
//
// Reference behaviour: ComputeMG.cpp:64-102 from that level down.
#include "coarse.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <cstring>

namespace hpcgx
{

constexpr int COARSE_TEAMS = 4;               // see coarse_symgs
// threads of a team, the most rows of a step: as many as leave a row's operands
// in registers (FP64 takes 153 of the 168 that 12 waves may have, mixed 94 of 128;
// no scratch)
template <typename XT>
constexpr int coarse_team() { return sizeof(XT) == 8 ? 192 : 256; }
template <typename XT>
constexpr int coarse_bs() { return COARSE_TEAMS * coarse_team<XT>(); }
constexpr size_t COARSE_LDS = 156 << 10;      // of the CU's 160 KB
constexpr int GROUPS = (W + 3) / 4;           // slots in groups of four: [4g, 4g + 4)

// the descriptions are read as constant memory: scalar loads, also after stores
typedef const __attribute__((address_space(4))) CoarseLevel ConstLevel;
typedef const __attribute__((address_space(4))) CoarseStep ConstStep;

enum CoarseKind : int
{
    CK_FWD,        // x = (r - A x) / d
    CK_BWD,        // x = (t - A x) / d
    CK_BWD_ZERO,   // x = (x d - A x) / d
    CK_BWD_ZERO_U, // s = x d - A x, t = x d - s, x = (s - B x) / d
    CK_FWD_T,      // t = r - A x, x = (t - B x) / d
    CK_FWD_U       // u = t, t = r - A x, x = (t - u - B x) / d
};

// One row's operands: the groups of its first sum, then those of its second.
constexpr int COARSE_GROUPS = 10;

template <typename VT, typename XT>
struct CoarseRow
{
    VT a[COARSE_GROUPS][4];
    uint2 at[COARSE_GROUPS];   // LDS offsets, 16 bits each
    XT r;                      // rhs, one of the two: no conversion before it has arrived
    double r64;
    VT d;
};

// Where a step's groups lie: pointers to their first slot's values and to their
// columns, both of the level's row 0 (uniform, advanced from group to group).
struct GroupPtr
{
    const char* val;
    const char* at;
    int slot;         // the group's first slot
};

// The groups of a step, one after the other; the recursion keeps every register
// index static and leaves at the last group.  From J = na on they are the second
// sum's (`b`).  vrow and irow: the row's byte offsets.
template <int J, typename VT, typename XT>
__device__ __forceinline__ void load_groups(GroupPtr g, GroupPtr b, int na, int n, int at_bytes, uint32_t vrow,
                                            uint32_t irow, CoarseRow<VT, XT>& o)
{
    constexpr int SLOT = (int)(ELL_SLICE * sizeof(VT));
    if constexpr(J < COARSE_GROUPS)
        if(J < n)
        {
            if(J == na) g = b;
            o.at[J] = *(const uint2*)(g.at + irow);
            const char* v = g.val + vrow;
            o.a[J][0] = *(const VT*)v;
            o.a[J][1] = *(const VT*)(v + SLOT);
            o.a[J][2] = *(const VT*)(v + 2 * SLOT);
            // the last group has three slots; its fourth, whose x is the zero, reads the third's value again
            o.a[J][3] = *(const VT*)(g.val + (g.slot + 3 < W ? 3 * SLOT : 2 * SLOT) + vrow);
            g.val += 4 * SLOT;
            g.at += at_bytes;
            g.slot += 4;
            load_groups<J + 1, VT, XT>(g, b, na, n, at_bytes, vrow, irow, o);
        }
}

template <typename VT>
__device__ __forceinline__ GroupPtr group_ptr(ConstLevel& L, int gv, int gi)
{
    return GroupPtr{(const char*)L.val + gv * (int)(4 * ELL_SLICE * sizeof(VT)), (const char*)L.at + gi * L.m * 8, 4 * gv};
}

// x of a group's slots
template <typename XT>
struct Quad
{
    XT x[4];
    __device__ __forceinline__ void read(const char* xs, uint2 at)
    {
        x[0] = *(const XT*)(xs + (at.x & 0xffffu));
        x[1] = *(const XT*)(xs + (at.x >> 16));
        x[2] = *(const XT*)(xs + (at.y & 0xffffu));
        x[3] = *(const XT*)(xs + (at.y >> 16));
    }
};

// s -= a x over the operands' groups [J, n); x0 and x1 hold the x of groups J and
// J + 1, read two groups ahead of their use
template <int J, typename VT, typename XT>
__device__ __forceinline__ void sum_from(const char* xs, int n, const CoarseRow<VT, XT>& o, const Quad<XT>& x0,
                                         const Quad<XT>& x1, XT& s)
{
    if constexpr(J < COARSE_GROUPS)
        if(J < n)
        {
            Quad<XT> x2;
            if constexpr(J + 2 < COARSE_GROUPS)
                if(J + 2 < n) x2.read(xs, o.at[J + 2]);
#pragma unroll
            for(int p = 0; p < 4; ++p) s = fmaT(-cvt<XT>(o.a[J][p]), x0.x[p], s);
            sum_from<J + 1, VT, XT>(xs, n, o, x1, x2, s);
        }
}

// s -= a x over the operands' groups [j0, n)
template <int J, typename VT, typename XT>
__device__ __forceinline__ void sum_groups(const char* xs, int j0, int n, const CoarseRow<VT, XT>& o, XT& s)
{
    if constexpr(J < COARSE_GROUPS)
    {
        if(J < j0)
        {
            sum_groups<J + 1, VT, XT>(xs, j0, n, o, s);
            return;
        }
        if(J < n)
        {
            Quad<XT> x0, x1;
            x0.read(xs, o.at[J]);
            if constexpr(J + 1 < COARSE_GROUPS)
                if(J + 1 < n) x1.read(xs, o.at[J + 1]);
            sum_from<J, VT, XT>(xs, n, o, x0, x1, s);
        }
    }
}

// How a level's steps are run
enum CoarseMode : int
{
    CM_PLAIN,   // no CK_FWD_T among them
    CM_ROWS,    // CK_FWD_T takes the diagonal of the row, as row_fwd_full does
    CM_USED     // every sum over its used slots alone
};

// The sum over the groups' used slots, straight from memory.
template <typename VT, typename XT>
__device__ __forceinline__ XT sum_used(ConstLevel& L, const char* xs, int gv, int gi, int n, int row, XT s)
{
    const uint32_t unused = (uint32_t)L.m * (uint32_t)sizeof(XT);
#pragma unroll 1
    for(int p = 0; p < 4 * n; ++p)
    {
        const uint32_t at = ((const uint16_t*)(L.at + (int64_t)(gi + p / 4) * L.m + row))[p % 4];
        if(at != unused) s = fmaT(-cvt<XT>(((const VT*)L.val)[ell_at(4 * gv + p, row)]), *(const XT*)(xs + at), s);
    }
    return s;
}

template <int MODE, typename VT, typename XT>
__device__ __forceinline__ void coarse_load(ConstLevel& L, const void* r, bool r_f64, const CoarseStep& S, int row,
                                            CoarseRow<VT, XT>& o)
{
    if constexpr(MODE != CM_USED)
        load_groups<0, VT, XT>(group_ptr<VT>(L, S.va, S.ia), group_ptr<VT>(L, S.vb, S.ib), S.na, S.na + S.nb, 8 * L.m,
                               (uint32_t)(ell_at(0, row) * sizeof(VT)), 8u * (uint32_t)row, o);
    if(MODE != CM_PLAIN && S.kind == CK_FWD_T)
        o.d = ((const VT*)L.val)[ell_at(L.diag_idx[row], row)];
    else
        o.d = ((const VT*)L.dg)[row];
    if(S.kind == CK_FWD || S.kind >= CK_FWD_T)
    {
        if(r_f64)
            o.r64 = ((const double*)r)[row];
        else
            o.r = ((const XT*)r)[row];
    }
}

// nan becomes NaN with a sum that is one
template <int MODE, typename VT, typename XT>
__device__ __forceinline__ void coarse_compute(ConstLevel& L, char* xs, XT* ts, bool r_f64, const CoarseStep& S, int row,
                                               const CoarseRow<VT, XT>& o, XT& nan)
{
#pragma clang fp contract(off)
    XT* mine = (XT*)xs + row;
    const XT d = cvt<XT>(o.d);
    XT s = r_f64 ? (XT)o.r64 : o.r, u = 0;
    if(S.kind == CK_BWD) s = ts[row];
    if(S.kind == CK_BWD_ZERO || S.kind == CK_BWD_ZERO_U) s = *mine * d;
    if(S.kind == CK_FWD_U) u = ts[row];
    const XT s0 = s;
    if constexpr(MODE == CM_USED)
        s = sum_used<VT, XT>(L, xs, S.va, S.ia, S.na, row, s);
    else
        sum_groups<0, VT, XT>(xs, 0, S.na, o, s);
    if(S.kind >= CK_BWD_ZERO_U)
    {
        ts[row] = S.kind == CK_BWD_ZERO_U ? s0 - s : s;
        if(S.kind == CK_FWD_U) s = s - u;
        if constexpr(MODE == CM_USED)
            s = sum_used<VT, XT>(L, xs, S.vb, S.ib, S.nb, row, s);
        else
            sum_groups<0, VT, XT>(xs, S.na, S.na + S.nb, o, s);
    }
    // a multiply-add a row; a look at each sum on the spot made 64^3 mixed 1.5% slower
    nan = fmaT((XT)0, s, nan);
    *mine = s / d;
}

__device__ __forceinline__ CoarseStep step_at(ConstStep* s)
{
    return CoarseStep{s->kind, s->off, s->n, s->va, s->ia, s->na, s->vb, s->ib, s->nb};
}

// A symmetric Gauss-Seidel sweep's steps [k0, k1).  The teams of the workgroup
// take them in turn; a barrier ends every step.  A team issues the loads of its
// next step right after it has computed one, T - 1 barriers ahead of their use.
// Every wave passes n = k1 - k0 barriers.
template <int MODE, typename VT, typename XT>
__device__ __forceinline__ void coarse_symgs(ConstLevel& L, char* lds, const void* r, bool r_f64, int k0, int k1, XT& nan)
{
    constexpr int T = COARSE_TEAMS;
    const int team = __builtin_amdgcn_readfirstlane((int)threadIdx.x / coarse_team<XT>());
    const int lane = (int)threadIdx.x % coarse_team<XT>();
    const int wave = __builtin_amdgcn_readfirstlane(lane) & ~63;
    char* xs = lds + L.lds_x;
    XT* ts = (XT*)(lds + L.lds_t);
    ConstStep* steps = (ConstStep*)L.steps + k0;
    const int n = k1 - k0;
    int passed = 0;   // barriers
    CoarseStep next = step_at(steps + min(team, n - 1));
#pragma unroll 1
    for(int k = team; k < n; k += T)
    {
        const CoarseStep S = next;
        CoarseRow<VT, XT> o;
        // threads past the step's rows load its last row and store nothing; waves
        // past them do neither
        const bool any = wave < S.n;
        if(any) coarse_load<MODE, VT, XT>(L, r, r_f64, S, S.off + min(lane, S.n - 1), o);
        next = step_at(steps + min(k + T, n - 1));
#pragma unroll 1
        for(; passed < k; ++passed) __syncthreads();
        if(any && lane < S.n) coarse_compute<MODE, VT, XT>(L, xs, ts, r_f64, S, S.off + lane, o, nan);
        __syncthreads();
        ++passed;
    }
#pragma unroll 1
    for(; passed < n; ++passed) __syncthreads();
}

// rc = the residual at the injected rows (row_restrict), into the next level's r
template <typename VT, typename XT>
__device__ __forceinline__ void coarse_restrict(ConstLevel& L, ConstLevel& C, char* lds, const void* r, bool r_f64,
                                                bool used, XT& nan)
{
    const int mc = L.mc, m = L.m;
    const char* xs = lds + L.lds_x;
    for(int k = threadIdx.x; k < mc; k += coarse_bs<XT>())
    {
        const int row = L.f2c_fine[k];
        XT s = r_f64 ? (XT)((const double*)r)[row] : ((const XT*)r)[row];
        if(used)
            s = sum_used<VT, XT>(L, xs, 0, SEC_ROW * GROUPS, GROUPS, row, s);
        else
        {
            CoarseRow<VT, XT> o;
            const GroupPtr g = group_ptr<VT>(L, 0, SEC_ROW * GROUPS);
            load_groups<0, VT, XT>(g, g, GROUPS, GROUPS, 8 * m, (uint32_t)(ell_at(0, row) * sizeof(VT)),
                                   8u * (uint32_t)row, o);
            sum_groups<0, VT, XT>(xs, 0, GROUPS, o, s);
        }
        nan = fmaT((XT)0, s, nan);
        ((XT*)C.r)[L.f2c_coarse[k]] = s;
    }
    __syncthreads();
}

template <typename VT, typename XT>
__device__ __forceinline__ void coarse_vcycle(const CoarseRun& R, char* lds)
{
    ConstLevel* lv = (ConstLevel*)R.lv;
    // the zero that unused slots read
    for(int l = threadIdx.x; l < R.nl; l += coarse_bs<XT>()) ((XT*)(lds + R.lv[l].lds_x))[R.lv[l].m] = 0;
    __syncthreads();
    XT nan = 0;
    bool used = false;
    // down, then up again; the bottom is its own way up
#pragma unroll 1
    for(int v = 0; v < 2 * R.nl - 1; ++v)
    {
        const bool up = v >= R.nl;
        const int l = up ? 2 * R.nl - 2 - v : v;
        const bool bottom = l + 1 == R.nl;
        ConstLevel& L = lv[l];
        XT* xs = (XT*)(lds + L.lds_x);
        const void* r = l == 0 ? R.r : L.r;
        const bool r64 = sizeof(XT) < sizeof(double) && l == 0 && R.r_f64;
        if(up)
        {
            const XT* xc = (const XT*)(lds + lv[l + 1].lds_x);
            const int mc = L.mc;
            for(int k = threadIdx.x; k < mc; k += coarse_bs<XT>())
            {
                const int f = L.f2c_fine[k];
                xs[f] = xs[f] + xc[L.f2c_coarse[k]];
            }
            __syncthreads();
        }
        const int k0 = up ? L.npre : 0, k1 = up ? L.npre + L.npost : L.npre;
        if(used)
            coarse_symgs<CM_USED, VT, XT>(L, lds, r, r64, k0, k1, nan);
        else if(up && L.whole_rows)
            coarse_symgs<CM_ROWS, VT, XT>(L, lds, r, r64, k0, k1, nan);
        else
            coarse_symgs<CM_PLAIN, VT, XT>(L, lds, r, r64, k0, k1, nan);
        if(!up && !bottom) coarse_restrict<VT, XT>(L, lv[l + 1], lds, r, r64, used, nan);
        if(up || bottom)
        {
            // before the result is written: r may be x
            if(l == 0 && !used && __syncthreads_or(nan != nan))
            {
                used = true;
                v = -1;
                continue;
            }
            XT* x = (XT*)(l == 0 ? R.x : L.x);
            const int m = L.m;
            for(int i = threadIdx.x; i < m; i += coarse_bs<XT>()) x[i] = xs[i];
        }
    }
}

template <typename VT, typename XT>
__global__ __launch_bounds__(coarse_bs<XT>()) void k_coarse(CoarseRun run)
{
    if(gated(run.gate)) return;
    extern __shared__ __align__(16) char coarse_lds_mem[];
    coarse_vcycle<VT, XT>(run, coarse_lds_mem);
}

template <typename VT, typename XT>
__global__ __launch_bounds__(coarse_bs<XT>()) void kb_coarse(const CoarseRun* __restrict__ runs)
{
    const CoarseRun run = runs[blockIdx.x];
    if(gated(run.gate)) return;
    extern __shared__ __align__(16) char coarse_lds_mem[];
    coarse_vcycle<VT, XT>(run, coarse_lds_mem);
}

// LDS offsets of a level's columns by section: [section][group][row][4]
__global__ __launch_bounds__(256) void k_coarse_columns(int m, int xbytes, const int32_t* __restrict__ col,
                                                        const int32_t* __restrict__ desc, uint16_t* __restrict__ at)
{
    const int row = blockIdx.x * 256 + threadIdx.x;
    if(row >= m) return;
    const int32_t ds = desc[row];
    for(int p = 0; p < 4 * GROUPS; ++p)
    {
        const int c = p < W ? col[ell_at(p, row)] : -1;
        const bool up = p < W && p >= desc_upper(ds), tail = p < W && p >= desc_tail(ds);
        const bool in[SEC_COUNT] = {p < desc_diag(ds), up, up && !tail, tail, p <= desc_diag(ds) || up};
        for(int s = 0; s < SEC_COUNT; ++s)
            at[(((int64_t)s * GROUPS + p / 4) * m + row) * 4 + p % 4] = (uint16_t)((in[s] ? c : m) * xbytes);
    }
}

// ---------------------------------------------------------------------------
// host

// x and the zero behind it
static size_t x_bytes(const Level& L, Prec prec)
{
    return ((size_t)(L.m + 1) * (prec == PREC_F64 ? 8 : 4) + 15) / 16 * 16;
}

// The steps of a level's smoothing: forward over the colours, back from the
// last but one, each colour's rows `team` at a time.  The last colour has no
// upper entries and no backward visit.  False: a step has more groups than a
// thread holds (colourings of many colours, with wide windows on both sides).
static bool add_steps(const Level& L, int team, bool post, bool keep_u, std::vector<CoarseStep>& out)
{
    const int n = L.ncolors;
    for(int v = 0; v < 2 * n - 1; ++v)
    {
        const bool fwd = v < n;
        const int c = fwd ? v : 2 * n - 2 - v;
        const int lower = (L.win[WIN_LOWER][c] + 3) / 4;
        const int upper = (W - L.win[WIN_UPPER][c]) / 4, tail = (W - L.win[WIN_TAIL][c]) / 4;
        CoarseStep s{};
        auto first = [&](int sec, int g0, int g1) { s.va = g0, s.ia = sec * GROUPS + g0, s.na = g1 - g0; };
        auto second = [&](int sec, int g0, int g1) { s.vb = g0, s.ib = sec * GROUPS + g0, s.nb = g1 - g0; };
        if(fwd)
        {
            s.kind = !post || c == n - 1 ? CK_FWD : L.u_ok ? CK_FWD_U : CK_FWD_T;
            first(SEC_LOWER, 0, lower);
            if(s.kind == CK_FWD_U) second(SEC_TAIL, tail, L.win[WIN_TAIL][c] ? GROUPS : tail);
            if(s.kind == CK_FWD_T) second(SEC_UPPER, upper, L.win[WIN_UPPER][c] ? GROUPS : upper);
        }
        else
        {
            s.kind = post ? CK_BWD : keep_u ? CK_BWD_ZERO_U : CK_BWD_ZERO;
            first(keep_u ? SEC_MID : SEC_UPPER, upper, L.win[WIN_UPPER][c] ? GROUPS : upper);
            if(keep_u) second(SEC_TAIL, tail, L.win[WIN_TAIL][c] ? GROUPS : tail);
        }
        if(s.na + s.nb > COARSE_GROUPS) return false;
        for(int i = 0; i < L.sizes[c]; i += team)
        {
            s.off = L.offsets[c] + i;
            s.n = std::min(team, L.sizes[c] - i);
            out.push_back(s);
        }
    }
    return true;
}

static int build_plan(Problem& P, Prec prec)
{
    CoarsePlan& C = P.coarse[prec];
    const int nl = P.nlevels;
    const int team = prec == PREC_F64 ? coarse_team<double>() : coarse_team<float>();
    // from the bottom up, while a level's offsets fit 16 bits and the run's x and t
    // the LDS
    size_t at = 0, ncol = 0;
    std::vector<CoarseLevel> h;
    std::vector<CoarseStep> steps;
    std::vector<size_t> first_step, cols;
    C.first = nl;
    for(int l = nl - 1; l >= 0; --l)
    {
        const Level& L = P.L[l];
        const size_t xb = x_bytes(L, prec), s0 = steps.size();
        const bool bottom = l + 1 == nl;
        if(xb > (64 << 10) || at + 2 * xb > COARSE_LDS) break;
        CoarseLevel c{};
        bool ok = add_steps(L, team, false, !bottom && L.u_ok, steps);
        c.npre = (int)(steps.size() - s0);
        if(!bottom) ok = ok && add_steps(L, team, true, false, steps);
        c.npost = (int)(steps.size() - s0) - c.npre;
        if(!ok)
        {
            steps.resize(s0);
            break;
        }
        c.lds_x = (int)at;
        c.lds_t = (int)(at + xb);
        at += 2 * xb;   // the bottom's t stays unused
        h.insert(h.begin(), c);
        first_step.insert(first_step.begin(), s0);
        cols.insert(cols.begin(), ncol);
        ncol += (size_t)SEC_COUNT * GROUPS * 4 * L.m;
        C.lds[l] = at;
        C.first = l;
    }
    const int nc = nl - C.first;
    if(nc == 0) return 0;
    // one allocation: columns, steps, descriptions
    const CoarseLayout lay = coarse_layout(ncol, steps.size(), nc);
    HPCGX_HIP(hipMalloc(&C.mem, lay.bytes));
    C.bytes = lay.bytes;
    char* mem = (char*)C.mem;
    for(int j = 0; j < nc; ++j)
    {
        const int l = C.first + j;
        const Level& L = P.L[l];
        const LevelVecs& V = prec == PREC_F64 ? P.v64[l] : P.v32[l];
        h[j].val = prec == PREC_F64 ? (const void*)L.ell_val : (const void*)L.ell_h;
        h[j].dg = prec == PREC_F64 ? (const void*)L.diag64 : (const void*)L.diag_h;
        h[j].diag_idx = L.diag_idx;
        h[j].at = (const uint2*)((uint16_t*)mem + cols[j]);
        h[j].f2c_fine = L.f2c_fine;
        h[j].f2c_coarse = L.f2c_coarse;
        h[j].steps = (const CoarseStep*)(mem + lay.steps) + first_step[j];
        h[j].r = V.r;
        h[j].x = V.x;
        h[j].m = (int)L.m;
        h[j].whole_rows = !L.u_ok;
        h[j].mc = j + 1 < nc ? (int)L.mc : 0;
        hipLaunchKernelGGL(k_coarse_columns, dim3((unsigned)ceil_div(L.m, 256)), dim3(256), 0, P.s, (int)L.m,
                           prec == PREC_F64 ? 8 : 4, L.ell_col, L.desc, (uint16_t*)mem + cols[j]);
        HPCGX_HIP(hipGetLastError());
    }
    std::vector<char>& up = C.upload;
    up.resize(lay.bytes - lay.steps);
    std::memcpy(up.data(), steps.data(), sizeof(CoarseStep) * steps.size());
    std::memcpy(up.data() + (lay.levels - lay.steps), h.data(), sizeof(CoarseLevel) * nc);
    HPCGX_HIP(hipMemcpyAsync(mem + lay.steps, up.data(), up.size(), hipMemcpyHostToDevice, P.s));
    C.lv = (CoarseLevel*)(mem + lay.levels);
    return 0;
}

int coarse_build(Problem& P)
{
    if(P.has_f64) HPCGX_TRY(build_plan(P, PREC_F64));
    if(P.has_mixed) HPCGX_TRY(build_plan(P, PREC_MIXED));
    return 0;
}

void coarse_free(Problem& P)
{
    for(CoarsePlan& C : P.coarse)
    {
        if(C.mem) (void)hipFree(C.mem);
        C = CoarsePlan();
    }
}

int coarse_first(const Problem& P, Prec prec)
{
    const int rows = P.coarse_rows < 0 ? COARSE_ROWS[prec] : P.coarse_rows;
    int l = P.nlevels;
    while(l > 0 && l - 1 >= P.coarse[prec].first && P.L[l - 1].m <= rows && !P.L[l - 1].exposed) --l;
    return l;
}

CoarseRun coarse_run(const Problem& P, int l, Prec prec, const void* r, bool r_f64, void* x, const int* gate)
{
    const CoarsePlan& C = P.coarse[prec];
    return CoarseRun{C.lv + (l - C.first), P.nlevels - l, r_f64 && prec != PREC_F64, r, x, gate};
}

// dynamic LDS above 64 KB has to be asked for
template <typename K>
static int allow_lds(K kernel)
{
    HPCGX_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)COARSE_LDS));
    return 0;
}

int launch_coarse(const CoarseRun& run, Prec prec, size_t lds, hipStream_t s)
{
    if(prec == PREC_F64)
    {
        HPCGX_TRY(allow_lds(k_coarse<double, double>));
        hipLaunchKernelGGL((k_coarse<double, double>), dim3(1), dim3(coarse_bs<double>()), lds, s, run);
    }
    else
    {
        HPCGX_TRY(allow_lds(k_coarse<__half, float>));
        hipLaunchKernelGGL((k_coarse<__half, float>), dim3(1), dim3(coarse_bs<float>()), lds, s, run);
    }
    HPCGX_HIP(hipGetLastError());
    return 0;
}

int launch_coarse_batch(const CoarseRun* runs, int n, Prec prec, size_t lds, hipStream_t s)
{
    if(prec == PREC_F64)
    {
        HPCGX_TRY(allow_lds(kb_coarse<double, double>));
        hipLaunchKernelGGL((kb_coarse<double, double>), dim3((unsigned)n), dim3(coarse_bs<double>()), lds, s, runs);
    }
    else
    {
        HPCGX_TRY(allow_lds(kb_coarse<__half, float>));
        hipLaunchKernelGGL((kb_coarse<__half, float>), dim3((unsigned)n), dim3(coarse_bs<float>()), lds, s, runs);
    }
    HPCGX_HIP(hipGetLastError());
    return 0;
}

}  // namespace hpcgx
