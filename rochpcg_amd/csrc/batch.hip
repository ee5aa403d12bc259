// batch.hip -- batched solves of many independent, unevenly sized HPCG
// problems.  Each problem keeps its own hierarchy, vectors, reduction scratch
// and CG scalars (a Problem); the V-cycle and the CG iteration are issued as
// one launch per (operator, level, colour) covering every problem, so a whole
// batched iteration is ~105 launches whatever the number of problems, and is
// captured once as a hipGraph.  Blocks map to (problem, row block) through a
// segment table in device memory (the segment records, then the segment of
// every block); a problem's segments return at once after its own
// convergence flag is set.
//
// Per-row arithmetic is shared with the single-problem kernels
// (kernels.hpp), so each problem computes exactly what it would alone, up to
// the grouping of the dot-product partials.
#include "batch.hpp"
#include "batch_rows.hpp"
#include "kernels.hpp"
#include "setup.hpp"

#include <algorithm>
#include <cstring>
#include <functional>

namespace hpcgx
{

// the fold of a reducing launch, a block a problem: it folds the partials of the
// problem's segments (one per block of theirs), the first of which is folds[k]
template <int BS>
__global__ __launch_bounds__(BS) void kb_fold(const BSeg* __restrict__ segs, const int32_t* __restrict__ folds)
{
    const BSeg& S = segs[folds[blockIdx.x]];
    if(gated(S.gate)) return;
    fold_partials<BS>(S.ra.partial, S.nfold, S.ra);
}

template <typename XT, int BS>
__global__ __launch_bounds__(BS) void kb_prolong(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    const int64_t k = lb * BS + threadIdx.x;
    if(k >= S.size) return;
    const int64_t f = S.f2c_fine[k];
    XT* x = (XT*)S.x;
    x[f] = x[f] + ((const XT*)S.rc)[S.f2c_coarse[k]];
}

// vector segments: block lb of the segment handles elements [lb*chunk, ...)
#define BCHUNK()                                                   \
    const int64_t chunk_ = (S.size + S.nblk - 1) / S.nblk;         \
    const int64_t e0 = lb * chunk_;                                \
    const int64_t e1 = (e0 + chunk_ < S.size) ? e0 + chunk_ : S.size;

template <typename XT, typename YT, int BS>
__global__ __launch_bounds__(BS) void kb_dot(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCHUNK();
    const XT* a = (const XT*)S.a;
    const YT* bb = (const YT*)S.b;
    double acc = 0.0;
    for(int64_t i = e0 + threadIdx.x; i < e1; i += BS) acc = fmaT((double)bb[i], (double)a[i], acc);
    block_partial<BS>(acc, S.ra.partial, S.part0 + lb);
}

template <typename ZT, int BS>
__global__ __launch_bounds__(BS) void kb_cg_p(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCHUNK();
    const ZT* z = (const ZT*)S.a;
    double* p = (double*)S.w;
    const bool first = S.ra.sc->iter == 0;
    const double beta = S.ra.sc->beta;
    for(int64_t i = e0 + threadIdx.x; i < e1; i += BS) p[i] = first ? (double)z[i] : fmaT(beta, p[i], (double)z[i]);
}

template <int BS>
__global__ __launch_bounds__(BS) void kb_cg_xr(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCHUNK();
    const double* p = (const double*)S.a;
    const double* Ap = (const double*)S.b;
    double* x = (double*)S.x;
    double* r = (double*)S.w;
    const double alpha = S.ra.sc->alpha;
    double acc = 0.0;
    for(int64_t i = e0 + threadIdx.x; i < e1; i += BS)
    {
        const double rv = fmaT(-alpha, Ap[i], r[i]);
        r[i] = rv;
        x[i] = fmaT(alpha, p[i], x[i]);
        acc = fmaT(rv, rv, acc);
    }
    block_partial<BS>(acc, S.ra.partial, S.part0 + lb);
}

template <int BS>
__global__ __launch_bounds__(BS) void kb_copy(const BSeg* __restrict__ segs, int nseg)
{
    BSEG();
    BCHUNK();
    const double* a = (const double*)S.a;
    double* w = (double*)S.w;
    for(int64_t i = e0 + threadIdx.x; i < e1; i += BS) w[i] = a[i];
}

// w = a + beta*b (ComputeWAXPBY's alpha == 1 form)
template <int BS>
__global__ __launch_bounds__(BS) void kb_waxpby(const BSeg* __restrict__ segs, int nseg, double beta)
{
    BSEG();
    BCHUNK();
    const double* a = (const double*)S.a;
    const double* bb = (const double*)S.b;
    double* w = (double*)S.w;
    for(int64_t i = e0 + threadIdx.x; i < e1; i += BS) w[i] = fmaT(beta, bb[i], a[i]);
}
#undef BCHUNK

// The problems' CG scalars: a solve's start values, and a copy for the host.  One
// launch for the batch in place of a copy per problem (see batch_cg).
__global__ __launch_bounds__(64) void kb_reset_scalars(CGScalars* const* sc, int n, double tol, int max_iter)
{
    const int k = blockIdx.x * 64 + threadIdx.x;
    if(k >= n) return;
    CGScalars v{};
    v.tol = tol;
    v.max_iter = max_iter;
    *sc[k] = v;
}

__global__ __launch_bounds__(64) void kb_read_scalars(CGScalars* const* sc, int n, CGScalars* out)
{
    const int k = blockIdx.x * 64 + threadIdx.x;
    if(k < n) out[k] = *sc[k];
}

// ---------------------------------------------------------------------------
// launching a planned record

template <int BS>
static void launch_bs(const BLaunch& L, hipStream_t s)
{
    const dim3 g((unsigned)L.nblocks), b(BS);
    const BSeg* T = L.segs;
    const int n = L.nseg;
    const bool f64 = L.prec == PREC_F64;
    switch(L.kind)
    {
    case BK_PROLONG:
        if(f64)
            hipLaunchKernelGGL((kb_prolong<double, BS>), g, b, 0, s, T, n);
        else
            hipLaunchKernelGGL((kb_prolong<float, BS>), g, b, 0, s, T, n);
        break;
    case BK_DOT:
        if(!L.bf32)
            hipLaunchKernelGGL((kb_dot<double, double, BS>), g, b, 0, s, T, n);
        else
            hipLaunchKernelGGL((kb_dot<double, float, BS>), g, b, 0, s, T, n);
        break;
    case BK_CG_P:
        if(!L.bf32)
            hipLaunchKernelGGL((kb_cg_p<double, BS>), g, b, 0, s, T, n);
        else
            hipLaunchKernelGGL((kb_cg_p<float, BS>), g, b, 0, s, T, n);
        break;
    case BK_CG_XR: hipLaunchKernelGGL((kb_cg_xr<BS>), g, b, 0, s, T, n); break;
    case BK_COPY: hipLaunchKernelGGL((kb_copy<BS>), g, b, 0, s, T, n); break;
    case BK_WAXPBY: hipLaunchKernelGGL((kb_waxpby<BS>), g, b, 0, s, T, n, L.beta); break;
    }
}

static int launch(const BLaunch& L, hipStream_t s)
{
    if(L.kind == BK_COARSE) return launch_coarse_batch(L.runs, L.nseg, (Prec)L.prec, L.lds, s);
    if(L.nblocks == 0) return 0;
    if(L.kind <= BK_RESTRICT)
        HPCGX_TRY(L.pat ? launch_batch_rows<true>(L, s) : launch_batch_rows<false>(L, s));
    else if(L.block == 64)
        launch_bs<64>(L, s);
    else if(L.block == 128)
        launch_bs<128>(L, s);
    else
        launch_bs<256>(L, s);
    HPCGX_HIP(hipGetLastError());
    if(L.kind == BK_DOT || L.kind == BK_CG_XR || (L.kind == BK_SPMV && L.dot))
    {
        hipLaunchKernelGGL((kb_fold<FOLD_THREADS>), dim3((unsigned)L.nfolds), dim3(FOLD_THREADS), 0, s, L.segs, L.folds);
        HPCGX_HIP(hipGetLastError());
    }
    return 0;
}

// ---------------------------------------------------------------------------
// planning

struct Planner
{
    Batch& B;
    std::vector<BLaunch>* out;
    int prec;
    int next_bf32 = 0;   // the next vector launch reads an f32 z
    // slot windows of the next sweep launch (full rows unless set)
    int next_win = W, next_tail = W, next_all_u = 0;
    // rows per thread of the next sweep launch (2 needs even segment offsets and sizes)
    int next_rows = 1;
    // segments per problem of the next launch, and the one being filled
    int next_subs = 1, sub = 0;

    // widest window of kind `wk` of colour c on level l over the problems
    // that have the colour
    int widest(int l, int wk, int c)
    {
        int w = 0;
        for(Problem* P : B.probs)
            if(c < P->L[l].ncolors) w = std::max<int>(w, P->L[l].win[wk][c]);
        return w;
    }

    // append the launch (launch_end: or launches) whose segments are built by `fill(k, seg) -> bool`
    template <typename Fill>
    int add(int kind, int block, bool vector_kind, int r_f64, int dot, double beta, Fill&& fill)
    {
        std::vector<BSeg> segs;
        std::vector<size_t> prob;
        for(size_t k = 0; k < B.probs.size(); ++k)
            for(sub = 0; sub < next_subs; ++sub)
            {
                BSeg sg;
                std::memset(&sg, 0, sizeof(sg));
                sg.gate = &B.probs[k]->sc->done;
                if(!fill((int)k, sg) || sg.size <= 0) continue;
                segs.push_back(sg);
                prob.push_back(k);
            }
        BLaunch L;
        std::memset(&L, 0, sizeof(L));
        L.kind = kind;
        L.prec = prec;
        L.r_f64 = r_f64;
        L.dot = dot;
        L.block = block;
        L.beta = beta;
        L.bf32 = next_bf32;
        L.win = next_win;
        L.win_tail = next_tail;
        L.all_u = next_all_u;
        L.rows = launch_rows(segs.data(), segs.size(), next_rows);
        next_subs = 1;
        next_bf32 = 0;
        next_win = next_tail = W;
        next_all_u = 0;
        next_rows = 1;
        for(size_t j0 = 0, e; j0 < segs.size(); j0 = e)
        {
            e = launch_end(prob, j0);
            HPCGX_TRY(add_launch(L, segs.data() + j0, prob.data() + j0, e - j0, vector_kind));
        }
        return 0;
    }

    // append launch L over nseg segments
    int add_launch(BLaunch L, BSeg* segs, const size_t* prob, size_t nseg, bool vector_kind)
    {
        L.nseg = (int)nseg;
        L.nblocks = assign_blocks(segs, nseg, L.block, vector_kind, L.rows);
        L.pat = L.kind <= BK_RESTRICT;
        std::vector<int32_t> folds;
        // the segments of a problem follow each other: their partials too, and
        // the first folds them all
        for(size_t j = 0, first = 0; j < nseg; ++j)
        {
            if(prob[j] != prob[first]) first = j;
            if(j == first && segs[j].ra.partial) folds.push_back((int32_t)j);
            segs[j].part0 = segs[first].nfold;
            segs[first].nfold += segs[j].nblk;
            if(segs[j].ra.partial && segs[first].nfold > B.probs[prob[j]]->partial_cap)
            {
                set_error("batched reduction exceeds the partial capacity");
                return -2;
            }
            if(!segs[j].cols.pat) L.pat = 0;
            L.nrows += segs[j].size;
            if(segs[j].t) L.any_t = 1;
        }
        // the folds lie behind the map, whose last word seg_of reads whole
        const size_t folds_at = (table_bytes(nseg, L.nblocks) + 3) / 4 * 4;
        std::vector<char> h(folds_at + sizeof(int32_t) * folds.size());
        std::memcpy(h.data(), segs, sizeof(BSeg) * nseg);
        block_map(segs, nseg, reinterpret_cast<uint16_t*>(h.data() + sizeof(BSeg) * nseg));
        if(!folds.empty()) std::memcpy(h.data() + folds_at, folds.data(), sizeof(int32_t) * folds.size());
        HPCGX_HIP(hipMalloc((void**)&L.segs, h.size()));
        L.folds = (const int32_t*)((const char*)L.segs + folds_at);
        L.nfolds = (int)folds.size();
        B.tables.push_back(L.segs);
        HPCGX_HIP(hipMemcpy(L.segs, h.data(), h.size(), hipMemcpyHostToDevice));
        out->push_back(L);
        return 0;
    }

    RedArgs red(Problem* P, int op)
    {
        RedArgs ra;
        ra.partial = P->partial;
        ra.op = op;
        ra.sc = P->sc;
        ra.hist = P->hist;
        ra.hist_cap = P->hist_cap;
        ra.out = P->dout;
        ra.cap = P->partial_cap;
        return ra;
    }

    const void* vals(const Level& L) { return prec == PREC_F64 ? (const void*)L.ell_val : (const void*)L.ell_h; }
    const void* diags(const Level& L) { return prec == PREC_F64 ? (const void*)L.diag64 : (const void*)L.diag_h; }
    ColArgs columns(const Level& L, int c)
    {
        ColArgs a = L.cols(c);
        if(!L.use_pat()) a.pat = nullptr;
        return a;
    }
    LevelVecs* vecs(Problem* P) { return prec == PREC_F64 ? P->v64 : P->v32; }
    void* z(Problem* P) { return prec == PREC_F64 ? (void*)P->z64 : (void*)P->z32; }

    // The problems leave the launches together, at the first level that one
    // workgroup can take for each of them: a problem that left earlier would save
    // no launch and keep the others waiting (64 problems of 16^3 to 96^3 to 1e-9 in
    // FP64: 5% slower than without when each leaves at its own level, 1.3% faster
    // when all leave at the coarsest).
    int coarse_from()
    {
        int l = 0;
        for(const Problem* P : B.probs) l = std::max(l, coarse_first(*P, (Prec)prec));
        return l;
    }

    int64_t level_rows(int l)
    {
        int64_t m = 0;
        for(const Problem* P : B.probs) m += P->L[l].m;
        return m;
    }

    int block(int l) { return B.block[l] ? B.block[l] : default_block(level_rows(l)); }

    int max_colors(int l)
    {
        int n = 0;
        for(Problem* P : B.probs) n = std::max(n, P->L[l].ncolors);
        return n;
    }

    // one launch, a workgroup per problem, for the levels from l down
    int coarse(int l)
    {
        std::vector<CoarseRun> runs;
        BLaunch L;
        std::memset(&L, 0, sizeof(L));
        for(Problem* P : B.probs)
        {
            const LevelVecs& V = vecs(P)[l];
            runs.push_back(coarse_run(*P, l, (Prec)prec, l == 0 ? (const void*)P->r : V.r, l == 0, l == 0 ? z(P) : V.x,
                                      &P->sc->done));
            L.lds = std::max(L.lds, P->coarse[prec].lds[l]);
            L.bytes += vcycle_bytes(*P, l, prec != PREC_F64, false);
            L.stream_bytes += vcycle_bytes(*P, l, prec != PREC_F64, true);
        }
        L.kind = BK_COARSE;
        L.prec = prec;
        L.nseg = (int)runs.size();
        HPCGX_HIP(hipMalloc((void**)&L.runs, sizeof(CoarseRun) * runs.size()));
        B.tables.push_back(L.runs);
        HPCGX_HIP(hipMemcpy(L.runs, runs.data(), sizeof(CoarseRun) * runs.size(), hipMemcpyHostToDevice));
        out->push_back(L);
        return 0;
    }

    // the V-cycle from level l (ComputeMG.cpp:64-102), all problems in lockstep
    int mg(int l)
    {
        const int bs = block(l);
        const bool last = (l + 1 == B.nlevels);
        const int r64 = (l == 0) ? 1 : (prec == PREC_F64);
        if(l >= coarse_from()) return coarse(l);
        auto level_seg = [&](int k, BSeg& s, int c) {
            Problem* P = B.probs[k];
            const Level& L = P->L[l];
            if(c >= L.ncolors) return false;
            s.off = L.offsets[c];
            s.size = L.sizes[c];
            s.cols = columns(L, c);
            s.val = vals(L);
            s.dg = diags(L);
            s.r = (l == 0) ? (const void*)P->r : vecs(P)[l].r;
            s.x = (l == 0) ? z(P) : vecs(P)[l].x;
            return true;
        };
        const int C = max_colors(l);
        for(int c = 0; c < C; ++c)
        {
            next_win = widest(l, WIN_LOWER, c);
            next_rows = B.rows[l];
            HPCGX_TRY(add(BK_FWD_ZERO, bs, false, r64, 0, 0.0, [&](int k, BSeg& s) { return level_seg(k, s, c); }));
        }
        // the pre-smoother keeps its upper sums for the post-smoother where
        // the correction changes only last-colour rows (Level::u_ok)
        for(int c = C - 2; c >= 0; --c)
        {
            next_win = widest(l, WIN_UPPER, c);
            next_rows = B.rows[l];
            HPCGX_TRY(add(BK_BWD_ZERO, bs, false, r64, 0, 0.0, [&](int k, BSeg& s) {
                if(!(c <= B.probs[k]->L[l].ncolors - 2 && level_seg(k, s, c))) return false;
                if(!last && B.probs[k]->L[l].u_ok) s.t = vecs(B.probs[k])[l].t;
                return true;
            }));
        }
        if(last) return 0;
        HPCGX_TRY(add(BK_RESTRICT, bs, false, r64, 0, 0.0, [&](int k, BSeg& s) {
            Problem* P = B.probs[k];
            const Level& L = P->L[l];
            s.size = L.mc;
            s.cols = columns(L, L.ncolors - 1);
            if(!L.u_ok) s.cols.pat = nullptr;   // injected rows of several colours
            s.val = vals(L);
            s.f2c_fine = L.f2c_fine;
            s.f2c_coarse = L.f2c_coarse;
            s.r = (l == 0) ? (const void*)P->r : vecs(P)[l].r;
            s.x = (l == 0) ? z(P) : vecs(P)[l].x;
            s.rc = vecs(P)[l + 1].r;
            return true;
        }));
        HPCGX_TRY(mg(l + 1));
        HPCGX_TRY(add(BK_PROLONG, bs, false, r64, 0, 0.0, [&](int k, BSeg& s) {
            Problem* P = B.probs[k];
            const Level& L = P->L[l];
            s.size = L.mc;
            s.f2c_fine = L.f2c_fine;
            s.f2c_coarse = L.f2c_coarse;
            s.rc = vecs(P)[l + 1].x;
            s.x = (l == 0) ? z(P) : vecs(P)[l].x;
            return true;
        }));
        for(int c = 0; c < C; ++c)
        {
            bool all_u = true;
            for(Problem* P : B.probs)
                if(c < P->L[l].ncolors) all_u = all_u && c < P->L[l].ncolors - 1 && P->L[l].u_ok;
            if(all_u)
            {
                next_all_u = 1;
                next_win = widest(l, WIN_LOWER, c);
                next_tail = widest(l, WIN_TAIL, c);
            }
            next_rows = B.rows[l];
            HPCGX_TRY(add(BK_FWD_FULL, bs, false, r64, 0, 0.0, [&](int k, BSeg& s) {
                if(!level_seg(k, s, c)) return false;
                const bool before_last = c < B.probs[k]->L[l].ncolors - 1;
                s.t = before_last ? vecs(B.probs[k])[l].t : nullptr;
                s.use_u = before_last && B.probs[k]->L[l].u_ok;
                return true;
            }));
        }
        for(int c = C - 2; c >= 0; --c)
        {
            next_win = widest(l, WIN_UPPER, c);
            next_rows = B.rows[l];
            HPCGX_TRY(add(BK_BWD_FULL, bs, false, r64, 0, 0.0, [&](int k, BSeg& s) {
                if(!(c <= B.probs[k]->L[l].ncolors - 2 && level_seg(k, s, c))) return false;
                s.t = vecs(B.probs[k])[l].t;
                return true;
            }));
        }
        return 0;
    }

    int outer_spmv(bool dot, bool from_x, bool into_tmp)
    {
        next_subs = max_colors(0);   // one segment per colour: a block stages one colour's patterns
        // two rows a thread where one problem of as many rows has them
        // (default_shapes): 64 problems of 12.5M rows take 576 us in place of 645 in
        // FP64, 275 in place of 331 mixed
        next_rows = level_rows(0) > SMALL_ROWS ? 2 : 1;
        return add(BK_SPMV, block(0), false, 1, dot ? 1 : 0, 0.0, [&](int k, BSeg& s) {
            Problem* P = B.probs[k];
            const Level& L = P->L[0];
            if(sub >= L.ncolors) return false;
            s.off = L.offsets[sub];
            s.size = L.sizes[sub];
            s.cols = columns(L, sub);
            s.val = vals(L);
            s.r = from_x ? (const void*)P->x : (const void*)P->p;
            s.x = into_tmp ? (void*)P->tmp : (void*)P->Ap;
            if(dot) s.ra = red(P, OP_PAP);
            return true;
        });
    }

    int vec(int kind, int op, std::function<void(Problem*, BSeg&)> set, double beta = 0.0)
    {
        return add(kind, RED_THREADS, true, 1, 0, beta, [&](int k, BSeg& s) {
            Problem* P = B.probs[k];
            s.size = P->L[0].m;
            set(P, s);
            if(op != OP_NONE) s.ra = red(P, op);
            return true;
        });
    }

    int true_residual(int op)
    {
        HPCGX_TRY(outer_spmv(false, true, true));
        HPCGX_TRY(vec(BK_WAXPBY, OP_NONE, [](Problem* P, BSeg& s) {
            s.a = P->b;
            s.b = P->tmp;
            s.w = P->r;
        }, -1.0));
        return vec(BK_DOT, op, [](Problem* P, BSeg& s) {
            s.a = P->r;
            s.b = P->r;
        });
    }
};

static int plan(Batch& B)
{
    if(B.probs.size() > MAX_SEGS)   // a segment each in the vector launches
    {
        set_error("too many problems in one batch");
        return -2;
    }
    for(int mode = 0; mode < 2; ++mode)
    {
        const bool mixed = mode == CG_MIXED;
        if(mixed ? !B.probs[0]->has_mixed : !B.probs[0]->has_f64) continue;
        const int prec = mixed ? PREC_MIXED : PREC_F64;
        // preamble (CG.cpp:133-137): p = x; Ap = A p; r = b - Ap; ||r||
        Planner pre{B, &B.pre[mode], prec};
        HPCGX_TRY(pre.vec(BK_COPY, OP_NONE, [](Problem* P, BSeg& s) {
            s.a = P->x;
            s.w = P->p;
        }));
        HPCGX_TRY(pre.outer_spmv(false, false, false));
        HPCGX_TRY(pre.vec(BK_WAXPBY, OP_NONE, [](Problem* P, BSeg& s) {
            s.a = P->b;
            s.b = P->Ap;
            s.w = P->r;
        }, -1.0));
        HPCGX_TRY(pre.vec(BK_DOT, OP_NORMR0, [](Problem* P, BSeg& s) {
            s.a = P->r;
            s.b = P->r;
        }));
        // one iteration (CG.cpp:150-171)
        Planner it{B, &B.iter[mode], prec};
        HPCGX_TRY(it.mg(0));
        it.next_bf32 = mixed;   // r (f64) . z (f32 in the mixed mode)
        HPCGX_TRY(it.vec(BK_DOT, OP_RTZ, [mixed](Problem* P, BSeg& s) {
            s.a = P->r;
            s.b = mixed ? (const void*)P->z32 : (const void*)P->z64;
        }));
        it.next_bf32 = mixed;
        HPCGX_TRY(it.vec(BK_CG_P, OP_NONE, [mixed](Problem* P, BSeg& s) {
            s.a = mixed ? (const void*)P->z32 : (const void*)P->z64;
            s.w = P->p;
            s.ra.sc = P->sc;
        }));
        HPCGX_TRY(it.outer_spmv(true, false, false));
        HPCGX_TRY(it.vec(BK_CG_XR, OP_NORMR, [](Problem* P, BSeg& s) {
            s.a = P->p;
            s.b = P->Ap;
            s.x = P->x;
            s.w = P->r;
        }));
    }
    B.planned = true;
    B.routes.clear();
    for(const Problem* P : B.probs) B.routes.push_back(P->routes);
    return 0;
}

// ---------------------------------------------------------------------------

static void free_plans(Batch& B)
{
    for(int g = 0; g < 2; ++g)
    {
        if(B.gexec[g]) (void)hipGraphExecDestroy(B.gexec[g]);
        if(B.graph[g]) (void)hipGraphDestroy(B.graph[g]);
        B.gexec[g] = nullptr;
        B.graph[g] = nullptr;
        B.pre[g].clear();
        B.iter[g].clear();
    }
    for(void* t : B.tables) (void)hipFree(t);
    B.tables.clear();
    B.planned = false;
}

// the plans as the problems' switches are now
static int ensure_plan(Batch& B)
{
    bool same = B.planned;
    for(size_t k = 0; same && k < B.probs.size(); ++k) same = B.probs[k]->routes == B.routes[k];
    if(same) return 0;
    HPCGX_HIP(hipStreamSynchronize(B.s));
    free_plans(B);
    const int rc = plan(B);
    if(rc) free_plans(B);
    return rc;
}

int batch_create(Batch*& out, int nprob, const int* dims, int nlevels, bool with_f64, bool with_mixed, hipStream_t s)
{
    out = nullptr;
    if(nprob < 1)
    {
        set_error("a batch needs at least one problem");
        return -2;
    }
    Batch* B = new Batch;
    B->nlevels = nlevels;
    if(s)
        B->s = s;
    else
    {
        if(hipStreamCreateWithFlags(&B->s, hipStreamNonBlocking) != hipSuccess)
        {
            set_error("cannot create the batch stream");
            delete B;
            return -1;
        }
        B->own_stream = true;
    }
    for(int k = 0; k < nprob; ++k)
    {
        Problem* P = nullptr;
        int rc = problem_create(P, dims[3 * k], dims[3 * k + 1], dims[3 * k + 2], nlevels, with_f64, with_mixed, B->s);
        if(rc)
        {
            batch_destroy(B);
            return rc;
        }
        B->probs.push_back(P);
    }
    std::vector<CGScalars*> sc;
    for(const Problem* P : B->probs) sc.push_back(P->sc);
    const size_t bytes = sizeof(CGScalars*) * sc.size();
    if(hipMalloc((void**)&B->sc, bytes) != hipSuccess ||
       hipMemcpy(B->sc, sc.data(), bytes, hipMemcpyHostToDevice) != hipSuccess ||
       hipHostMalloc((void**)&B->h_sc, 2 * sizeof(CGScalars) * sc.size(), hipHostMallocDefault) != hipSuccess ||
       hipEventCreateWithFlags(&B->read[0], hipEventDisableTiming) != hipSuccess ||
       hipEventCreateWithFlags(&B->read[1], hipEventDisableTiming) != hipSuccess)
    {
        set_error("cannot allocate the batch's scalars");
        batch_destroy(B);
        return -1;
    }
    out = B;
    return 0;
}

void batch_destroy(Batch* B)
{
    if(!B) return;
    if(B->s) (void)hipStreamSynchronize(B->s);
    free_plans(*B);
    for(Problem* P : B->probs) problem_destroy(P);
    if(B->sc) (void)hipFree(B->sc);
    if(B->h_sc) (void)hipHostFree(B->h_sc);
    for(hipEvent_t e : B->read)
        if(e) (void)hipEventDestroy(e);
    if(B->own_stream && B->s) (void)hipStreamDestroy(B->s);
    delete B;
}

int batch_set_block(Batch& B, int level, int block)
{
    if(level < 0 || level >= B.nlevels || (block != 64 && block != 128 && block != 256))
    {
        set_error("invalid level or block size");
        return -2;
    }
    B.block[level] = block;
    HPCGX_HIP(hipStreamSynchronize(B.s));
    free_plans(B);
    return 0;
}

int batch_set_rows(Batch& B, int level, int rows)
{
    if(level < 0 || level >= B.nlevels || (rows != 1 && rows != 2))
    {
        set_error("invalid level or rows per thread");
        return -2;
    }
    B.rows[level] = rows;
    HPCGX_HIP(hipStreamSynchronize(B.s));
    free_plans(B);
    return 0;
}

static int run_list(const std::vector<BLaunch>& v, hipStream_t s)
{
    for(const BLaunch& L : v) HPCGX_TRY(launch(L, s));
    return 0;
}

// algorithmic HBM bytes of one planned launch (the per-row model of iteration_bytes
// in solver.hip over the launch's rows): by the ELL's bytes, or (stream) what its
// kernel loads
static double launch_bytes(const BLaunch& L, bool stream)
{
    const bool f64 = L.prec == PREC_F64, pat = stream && L.pat;
    const double vb = f64 ? 8.0 : 2.0, xb = f64 ? 8.0 : 4.0, rb = L.r_f64 ? 8.0 : xb;
    const double slot = vb + (pat ? 0.0 : 4.0), head = pat ? 1.0 : 4.0, full = stream ? head : 0.0, n = (double)L.nrows;
    const double zb = L.bf32 ? 4.0 : 8.0;
    switch(L.kind)
    {
    case BK_SPMV: return n * (W * slot + full + 16.0);
    case BK_FWD_ZERO: return n * (window_slots(L.win) * slot + head + vb + rb + xb);
    case BK_BWD_ZERO: return n * (window_slots(L.win) * slot + head + vb + 2.0 * xb + (L.any_t ? xb : 0.0));
    case BK_FWD_FULL:
        if(L.all_u)
        {
            int na = 0, nb = 0;
            window_pair_slots(L.win, L.win_tail, &na, &nb);
            return n * ((na + nb) * slot + head + vb + rb + 3.0 * xb);
        }
        return n * (W * slot + full + rb + xb + (L.any_t ? xb : 0.0));
    case BK_BWD_FULL: return n * (window_slots(L.win) * slot + head + vb + 2.0 * xb);
    case BK_RESTRICT: return n * (W * slot + full + rb + 8.0 + xb);
    case BK_PROLONG: return n * (8.0 + 3.0 * xb);
    case BK_DOT: return n * (8.0 + zb);
    case BK_CG_P: return n * (zb + 16.0);
    case BK_CG_XR: return n * 48.0;
    case BK_COPY: return n * 16.0;
    case BK_WAXPBY: return n * 24.0;
    case BK_COARSE: return stream ? L.stream_bytes : L.bytes;
    }
    return 0.0;
}

// cg_begin's reset of every problem's scalars (tolerance 0: run max_iter)
static int reset_scalars(Batch& B, int max_iter, double tol)
{
    const int n = (int)B.probs.size();
    hipLaunchKernelGGL(kb_reset_scalars, dim3((unsigned)ceil_div(n, 64)), dim3(64), 0, B.s, B.sc, n, tol, max_iter);
    HPCGX_HIP(hipGetLastError());
    return 0;
}

// the scalars to the host's copy `slot`, there once B.read[slot] has come
static int read_scalars(Batch& B, int slot)
{
    const int n = (int)B.probs.size();
    hipLaunchKernelGGL(kb_read_scalars, dim3((unsigned)ceil_div(n, 64)), dim3(64), 0, B.s, B.sc, n, B.h_sc + slot * n);
    HPCGX_HIP(hipGetLastError());
    HPCGX_HIP(hipEventRecord(B.read[slot], B.s));
    return 0;
}

int batch_stream_bytes(Batch& B, int mode, double* bytes)
{
    if(mode != CG_F64 && mode != CG_MIXED)
    {
        set_error("invalid CG mode");
        return -2;
    }
    HPCGX_TRY(ensure_plan(B));
    if(B.iter[mode].empty())
    {
        set_error("the batch was built without the store this mode needs");
        return -2;
    }
    *bytes = 0.0;
    for(const BLaunch& L : B.iter[mode]) *bytes += launch_bytes(L, true);
    return 0;
}

int batch_profile(Batch& B, int mode, int iters, double* kind_ms, double* kind_bytes, double* iter_ms)
{
    if(mode != CG_F64 && mode != CG_MIXED)
    {
        set_error("invalid CG mode");
        return -2;
    }
    HPCGX_TRY(ensure_plan(B));
    const std::vector<BLaunch>& it = B.iter[mode];
    if(it.empty())
    {
        set_error("the batch was built without the store this mode needs");
        return -2;
    }
    if(iters < 1 || iters > B.probs[0]->hist_cap)
    {
        set_error("iteration count out of range");
        return -2;
    }
    HPCGX_TRY(reset_scalars(B, iters, 0.0));
    HPCGX_TRY(run_list(B.pre[mode], B.s));
    const size_t nl = it.size();
    std::vector<hipEvent_t> ev((size_t)iters * (nl + 1), nullptr);
    int rc = 0;
    for(auto& e : ev)
        if(hipEventCreate(&e) != hipSuccess)
        {
            set_error("hipEventCreate failed");
            rc = -1;
            break;
        }
    for(int i = 0; i < iters && !rc; ++i)
    {
        hipEvent_t* E = ev.data() + (size_t)i * (nl + 1);
        if(hipEventRecord(E[0], B.s) != hipSuccess) rc = -1;
        for(size_t j = 0; j < nl && !rc; ++j)
        {
            rc = launch(it[j], B.s);
            if(!rc && hipEventRecord(E[j + 1], B.s) != hipSuccess) rc = -1;
        }
    }
    if(!rc && hipStreamSynchronize(B.s) != hipSuccess)
    {
        set_error("stream synchronisation failed in a profiled batched run");
        rc = -1;
    }
    for(int k = 0; k < BK_COUNT; ++k)
    {
        kind_ms[k] = 0.0;
        kind_bytes[k] = 0.0;
    }
    // the coarse levels' launch, all kinds in one, counts as zero-guess forward sweeps
    auto kind_of = [&](size_t j) { return it[j].kind == BK_COARSE ? (int)BK_FWD_ZERO : it[j].kind; };
    double total = 0.0;
    if(!rc)
    {
        for(size_t j = 0; j < nl; ++j) kind_bytes[kind_of(j)] += launch_bytes(it[j], false);
        for(int i = 0; i < iters; ++i)
        {
            hipEvent_t* E = ev.data() + (size_t)i * (nl + 1);
            for(size_t j = 0; j < nl; ++j)
            {
                float ms = 0.f;
                if(hipEventElapsedTime(&ms, E[j], E[j + 1]) == hipSuccess) kind_ms[kind_of(j)] += ms;
            }
            float ms = 0.f;
            if(hipEventElapsedTime(&ms, E[0], E[nl]) == hipSuccess) total += ms;
        }
    }
    for(auto& e : ev)
        if(e) (void)hipEventDestroy(e);
    if(iter_ms) *iter_ms = total / iters;
    return rc;
}

int batch_cg(Batch& B, int mode, int max_iter, double tol, bool use_graph, int* niters, double* normr, double* normr0)
{
    if(mode != CG_F64 && mode != CG_MIXED)
    {
        set_error("invalid CG mode");
        return -2;
    }
    HPCGX_TRY(ensure_plan(B));
    if(B.iter[mode].empty())
    {
        set_error("the batch was built without the store this mode needs");
        return -2;
    }
    if(max_iter < 0 || max_iter > B.probs[0]->hist_cap)
    {
        set_error("max_iter out of range");
        return -2;
    }
    // per-problem scalars (cg_begin's reset)
    HPCGX_TRY(reset_scalars(B, max_iter, tol));
    HPCGX_TRY(run_list(B.pre[mode], B.s));
    if(use_graph && !B.gexec[mode])
    {
        HPCGX_HIP(hipStreamBeginCapture(B.s, hipStreamCaptureModeThreadLocal));
        const int rc = run_list(B.iter[mode], B.s);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(B.s, &g);
        if(rc || e != hipSuccess)
        {
            if(g) (void)hipGraphDestroy(g);
            if(rc) return rc;
            set_error(std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
            return -1;
        }
        e = hipGraphInstantiate(&B.gexec[mode], g, nullptr, nullptr, 0);
        if(e != hipSuccess)
        {
            (void)hipGraphDestroy(g);
            B.gexec[mode] = nullptr;
            set_error(std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
            return -1;
        }
        B.graph[mode] = g;
    }
    // The host looks at the convergence flags of the iteration before the one it
    // has queued last: the GPU always has work, and one iteration at most runs
    // after the last problem has converged (104 launches that find nothing to do,
    // 0.3 ms).  64 problems of 16^3 to 96^3 to 1e-9, against a look at every tenth
    // iteration with a copy per problem: 144.4 -> 136.7 ms in FP64, 84.5 -> 76.1
    // ms mixed.
    const size_t np = B.probs.size();
    bool all = false;
    for(int it = 0; it < max_iter && !all; ++it)
    {
        if(use_graph)
            HPCGX_HIP(hipGraphLaunch(B.gexec[mode], B.s));
        else
            HPCGX_TRY(run_list(B.iter[mode], B.s));
        if(tol <= 0.0) continue;
        HPCGX_TRY(read_scalars(B, it & 1));
        if(it == 0) continue;
        const int before = (it - 1) & 1;
        HPCGX_HIP(hipEventSynchronize(B.read[before]));
        all = true;
        for(size_t k = 0; k < np; ++k) all = all && B.h_sc[before * np + k].done;
    }
    HPCGX_TRY(read_scalars(B, 0));
    HPCGX_HIP(hipStreamSynchronize(B.s));
    const CGScalars* h = B.h_sc;
    for(size_t k = 0; k < B.probs.size(); ++k)
    {
        if(niters) niters[k] = h[k].iter;
        if(normr) normr[k] = h[k].normr;
        if(normr0) normr0[k] = h[k].normr0;
    }
    return 0;
}

}  // namespace hpcgx
