// lem_fa32.hip — flow accumulation of the FP32 form under single flow
// directions (CalcMFD with one receiver per cell, mfd_simple.cu:33-171) as
// exact integer subtree sums.
//
// With one receiver per cell the donor graph is a forest, and the
// reference's value of a completed cell, w + max(0, sum of donor fa), is the
// sum of w over the cell's subtree (every w >= 0, so the clamp never
// acts).  Each cell's weight is rounded once to a 64-bit fixed-point integer
// q = round(w * 2^F), with F chosen per DEM from its total runoff so that no
// sum can exceed 2^61; integer addition is associative, so the subtree sums
// are exact and do not depend on the order, the tiling or the other DEMs of
// an atlas.  The only rounding is that of q (relative 2^-F-ish, far below the
// FP32 form's 1e-6 bound) and of the final conversion to the float pair.
//
// Two passes over tiles of TW x TH cells with a small global solve between:
//   A. each tile sums its own subtrees in LDS by pointer doubling (round t
//      adds every cell's partial sum to its 2^t-th in-tile ancestor), which
//      also finds each cell's in-tile root, lists its exits (cells whose
//      receiver is in another tile) with their in-tile sums, and leaves every
//      in-tile sum in the cell's fa entry;
//   B. the exits form a forest of their own (an exit's parent is the exit
//      its receiver's in-tile path leads to); the same doubling over that
//      forest gives every exit its final value;
//   C. each tile adds the final values of the exits that flow into it along
//      their in-tile paths, and writes fa.
//
// Cycles: fd[outlet] = WEST can close a cycle through the outlet (the only
// possible one: every other link goes strictly downhill or down a plateau's
// distance field).  Cells on a cycle never complete in the reference and keep
// fa = w.  The outlet's link is cut and its west neighbour carries a tag of
// 2^62: tagged cells are exactly the path from the west neighbour to its
// root.  If the outlet is tagged, that path is the cycle (fa = w); otherwise
// the path lies downstream of the outlet and gets the outlet's sum added.
#include "lem_ctx.h"

#define FX_TAG (1ULL << 62)
#define FX_NONE 0xFFFFu   // no receiver
#define FX_EXIT 0xFFFEu   // the receiver is in another tile
#define FX_ROOT 0x8000u   // pass A: the pointer has reached the path's root
#define FX_CYCLE (1 << 30)   // in the exit count, more than any list holds: a tile's links close a cycle

// direction index of a single ESRI code, -1 for 0 or a multi-bit code
__device__ __forceinline__ int fx_dir(uint8_t code)
{
    switch (code) {
    case 64: return 0; case 128: return 1; case 1: return 2; case 2: return 3;
    case 4: return 4; case 8: return 5; case 16: return 6; case 32: return 7;
    default: return -1;
    }
}

__device__ __forceinline__ unsigned long long fx_quant(float w, int shift)
{
    return (unsigned long long)llrint(ldexp((double)w, shift));
}

__device__ __forceinline__ float2 fx_value(unsigned long long s, int shift)
{
    const double v = ldexp((double)s, -shift);
    const float hi = (float)v;
    return make_float2(hi, (float)(v - (double)hi));
}

// the tagged cell of a slot: the west neighbour of an outlet whose link to
// it exists (outlet valid, not in column 0, west neighbour valid)
__device__ __forceinline__ bool fx_tagged(long i, int W, const uint8_t *mask, int outlet)
{
    return outlet >= 1 && i == (long)outlet - 1 && (outlet % W) != 0 && mask[outlet] && mask[outlet - 1];
}

struct FxArgs {
    int W, H;
    const uint8_t *mask, *fd, *demid;
    const float *w;
    const DemScal *ds;
    const int *shift;            // per slot
    int nslot;
    // pass A outputs / pass C inputs (and the in-tile sums, in fa)
    int *exit_id;                // per cell (exits only)
    int *xroot;                  // per cell (tile border cells only): exit its in-tile path leads to, or -1
    unsigned long long *ex_val;  // per exit: in-tile sum (A), final value after the forest solve
    int *ex_recv;                // per exit: receiver cell
    int *ex_count;
    int ex_cap;
    // pass C outputs
    float2 *fa;
    int *tag_cell;
    unsigned long long *tag_sum;
    int *tag_count;
    int tag_cap;
    DemScal *dsw;
};

// n items of this thread appended to a global list with one atomic per
// block; returns this thread's first index (every thread must call it)
__device__ __forceinline__ int fx_block_append(int *counter, int n, int *s_wave, int *s_base)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int x = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
            const int cnt = s_wave[w];
            s_wave[w] = tot;
            tot += cnt;
        }
        *s_base = tot ? atomicAdd(counter, tot) : 0;
    }
    __syncthreads();
    const int pos = *s_base + s_wave[wave] + x - n;
    __syncthreads();
    return pos;
}

// padded (TW+2) x (TH+2) index of tile cell (lr, lc); the ring holds the
// neighbours in other tiles (or off the grid)
template <int TW> __device__ __forceinline__ int fx_pad(int lr, int lc) { return (lr + 1) * (TW + 2) + lc + 1; }

// A tile's directions, mask and links in LDS
template <int TW, int TH>
struct FxTile {
    static constexpr int NC = TW * TH, PER = NC / 256, PW = TW + 2, NP = (TW + 2) * (TH + 2);
    static constexpr int NPPER = (NP + 255) / 256, NB = 2 * TW + 2 * (TH - 2);
    static_assert(NC % 256 == 0 && NB <= 256 && NC <= (int)FX_ROOT, "tile shape");
    unsigned long long x[NC];
    uint16_t J[NC];   // pointer of the doubling (A); receiver in the tile, FX_EXIT or FX_NONE (C)
    uint8_t sfd[NP], smk[NP];
    int outlet[LEM_MAX_SLOTS + 1], shift[LEM_MAX_SLOTS + 1];   // per DEM
};

template <int TW, int TH> __device__ __forceinline__ void fx_slots(const FxArgs &a, FxTile<TW, TH> &T)
{
    for (int s = threadIdx.x; s < a.nslot; s += 256) {
        T.outlet[s] = a.ds[s].outlet;
        T.shift[s] = a.shift[s];
    }
}

// border cell k of a tile: the first and last row, then the two columns
template <int TW, int TH>
__device__ __forceinline__ void fx_border(int k, int &lr, int &lc)
{
    if (k < 2 * TW) {
        lr = k < TW ? 0 : TH - 1;
        lc = k < TW ? k : k - TW;
    } else {
        lr = 1 + ((k - 2 * TW) >> 1);
        lc = (k & 1) ? TW - 1 : 0;
    }
}

// receiver of tile cell (lr, lc), a mask cell
template <int TW, int TH>
__device__ __forceinline__ uint16_t fx_link(const FxTile<TW, TH> &T, int lr, int lc, bool is_outlet)
{
    const int p = fx_pad<TW>(lr, lc);
    const int d = fx_dir(T.sfd[p]);
    if (d < 0 || is_outlet || !T.smk[p + cdy(d) * FxTile<TW, TH>::PW + cdx(d)]) return FX_NONE;
    const int nr = lr + cdy(d), nc = lc + cdx(d);
    return nr >= 0 && nr < TH && nc >= 0 && nc < TW ? (uint16_t)(nr * TW + nc) : (uint16_t)FX_EXIT;
}

// Loads of both passes: directions and mask of the tile and its ring, each
// cell's slot and val(i) (kept by the caller in registers), with every load in
// flight before the first use.  Off-grid positions: no mask, no code.
template <int TW, int TH, typename V, class F>
__device__ __forceinline__ void fx_load(const FxArgs &a, int tx0, int ty0, FxTile<TW, TH> &T, V *v, int *slot, F &&val)
{
    typedef FxTile<TW, TH> FT;
    const int W = a.W, H = a.H;
    // offsets from the tile's first cell: 32 bits beside a uniform base (a
    // 64-bit address per load in flight would take half the registers)
    const long c0 = (long)ty0 * W + tx0;
    const uint8_t *fd0 = a.fd + c0, *mask0 = a.mask + c0, *dem0 = a.demid + c0;
    uint32_t vf[FT::NPPER], vm[FT::NPPER];   // 32-bit: byte registers would be packed, with a wait per load
#pragma unroll
    for (int q = 0; q < FT::NPPER; q++) {
        const int k = threadIdx.x + q * 256;
        const int ry = k / FT::PW - 1, rx = k % FT::PW - 1;
        const bool in = k < FT::NP && ty0 + ry >= 0 && ty0 + ry < H && tx0 + rx >= 0 && tx0 + rx < W;
        const int n = ry * W + rx;
        vf[q] = in ? fd0[n] : 0;
        vm[q] = in ? mask0[n] : 0;
    }
#pragma unroll
    for (int q = 0; q < FT::PER; q++) {
        const int li = threadIdx.x + q * 256;
        const int r = li / TW, col = li % TW;
        const int n = ty0 + r < H && tx0 + col < W ? r * W + col : 0;
        v[q] = val(c0, n);
        slot[q] = a.demid ? (int)dem0[n] : 0;
    }
#pragma unroll
    for (int q = 0; q < FT::NPPER; q++) {
        const int k = threadIdx.x + q * 256;
        if (k < FT::NP) {
            T.sfd[k] = vf[q];
            T.smk[k] = vm[q];
        }
    }
}

// Pass A.  After round t a cell holds the sum over the cells within 2^(t+1) - 1
// links upstream in the tile, and its pointer, kept in a register as well, is
// its 2^(t+1)-th ancestor or, marked FX_ROOT, the root of its path if that is
// nearer: such a cell has nothing more to add.
//
// Both passes are bound by the latency of what a tile waits for (loads, seven
// rounds here, a path of the tile's height or so there) and hide it with five
// and six tiles per compute unit.  One workgroup per tile: in a loop over
// tiles the compiler keeps every cell's offsets in registers across the loop
// (155 of them, three tiles per compute unit).  4096^2: 285 -> 176 us here
// (a second pointer array for the roots and a wait per cell's weight before)
// and 361 -> 120 us for pass C, which used to repeat the doubling and to look
// up a border cell's donors one after another.  Walks from the leaves, each
// link taken once, instead of the doubling: 409 us (one long river keeps the
// tile's other waves waiting).
template <int TW, int TH>
__global__ void __launch_bounds__(256, 5) k_fx_sums(FxArgs a)
{
    typedef FxTile<TW, TH> FT;
    __shared__ FT T;
    __shared__ int s_wave[4], s_base;
    const int W = a.W, H = a.H;
    const int ntx = (W + TW - 1) / TW;
    const int tx0 = (int)(blockIdx.x % ntx) * TW, ty0 = (int)(blockIdx.x / ntx) * TH;
    fx_slots(a, T);
    float w[FT::PER];
    int slot[FT::PER];
    fx_load<TW, TH>(a, tx0, ty0, T, w, slot, [&](long c0, int n) { return (a.w + c0)[n]; });
    __syncthreads();
    int nexit = 0;
    uint32_t exits = 0, cells = 0;   // of this thread's cells
    uint32_t jr[FT::PER];
#pragma unroll
    for (int q = 0; q < FT::PER; q++) {
        const int li = threadIdx.x + q * 256;
        const int lr = li / TW, lc = li % TW;
        uint32_t j = FX_NONE;
        unsigned long long v = 0;
        if (T.smk[fx_pad<TW>(lr, lc)]) {
            const long i = (long)(ty0 + lr) * W + tx0 + lc;
            const int outlet = T.outlet[slot[q]];
            cells |= 1u << q;
            v = fx_quant(w[q], T.shift[slot[q]]);
            if (fx_tagged(i, W, a.mask, outlet)) v += FX_TAG;
            j = fx_link(T, lr, lc, i == outlet);
            if (j == FX_EXIT) {
                nexit++;
                exits |= 1u << q;
            }
        }
        if (j >= FX_EXIT) j = FX_ROOT | (uint32_t)li;
        T.x[li] = v;
        T.J[li] = (uint16_t)j;
        jr[q] = j;
    }
    for (int t = 0;; t++) {
        __syncthreads();
        unsigned long long v[FT::PER];
        uint32_t jj[FT::PER];
        int act = 0;
#pragma unroll
        for (int q = 0; q < FT::PER; q++) {
            jj[q] = FX_ROOT;
            if (!(jr[q] & FX_ROOT)) {
                act = 1;
                v[q] = T.x[threadIdx.x + q * 256];
                jj[q] = T.J[jr[q]];
            }
        }
        if (!__syncthreads_or(act)) break;
        if ((1 << t) >= FT::NC) {   // no path in the tile is that long: a cycle
            if (threadIdx.x == 0) atomicOr(a.ex_count, FX_CYCLE);
            return;
        }
#pragma unroll
        for (int q = 0; q < FT::PER; q++) {
            if (jr[q] & FX_ROOT) continue;
            atomicAdd(&T.x[jr[q]], v[q]);
            jr[q] = jj[q];
            T.J[threadIdx.x + q * 256] = (uint16_t)jj[q];
        }
    }
    int k = fx_block_append(a.ex_count, nexit, s_wave, &s_base);
#pragma unroll
    for (int q = 0; q < FT::PER; q++) {
        const int li = threadIdx.x + q * 256;
        const int lr = li / TW, lc = li % TW;
        const int r = ty0 + lr, col = tx0 + lc;
        if (!((cells >> q) & 1)) continue;
        const long i = (long)r * W + col;
        const unsigned long long s = T.x[li];
        reinterpret_cast<unsigned long long *>(a.fa)[i] = s;
        if (lr == 0 || lr == TH - 1 || lc == 0 || lc == TW - 1) {
            // the root is an exit if its receiver is a mask cell (in
            // another tile) and its link is not cut
            const int root = jr[q] & (FX_ROOT - 1), rr = root / TW, rc = root % TW;
            const long ri = (long)(ty0 + rr) * W + tx0 + rc;
            const bool ex = fx_link(T, rr, rc, ri == T.outlet[slot[q]]) == FX_EXIT;
            a.xroot[i] = ex ? (int)ri : -1;
        }
        if (!((exits >> q) & 1)) continue;
        if (k < a.ex_cap) {
            const int d = fx_dir(T.sfd[fx_pad<TW>(lr, lc)]);
            a.exit_id[i] = k;
            a.ex_val[k] = s;
            a.ex_recv[k] = (int)((long)(r + cdy(d)) * W + (col + cdx(d)));
        }
        k++;
    }
}

// Pass C.  Each border cell with donors in other tiles adds their final values
// to every cell of its in-tile path, itself included.
template <int TW, int TH>
__global__ void __launch_bounds__(256, 5) k_fx_final(FxArgs a)
{
    typedef FxTile<TW, TH> FT;
    __shared__ FT T;
    const int W = a.W, H = a.H;
    const int ntx = (W + TW - 1) / TW;
    const int tx0 = (int)(blockIdx.x % ntx) * TW, ty0 = (int)(blockIdx.x / ntx) * TH;
    fx_slots(a, T);
    unsigned long long x[FT::PER];
    int slot[FT::PER];
    fx_load<TW, TH>(a, tx0, ty0, T, x, slot,
                    [&](long c0, int n) { return (reinterpret_cast<const unsigned long long *>(a.fa) + c0)[n]; });
    __syncthreads();
    // donors in other tiles of this thread's border cell: their exit
    // numbers in one wait, their values in another
    unsigned long long in = 0;
    int at = -1;
    if (threadIdx.x < FT::NB) {
        int lr, lc;
        fx_border<TW, TH>(threadIdx.x, lr, lc);
        const int p = fx_pad<TW>(lr, lc);
        if (T.smk[p]) {
            const long i = (long)(ty0 + lr) * W + tx0 + lc;
            const int out = T.outlet[a.demid ? (int)a.demid[i] : 0];
            int id[8];
#pragma unroll
            for (int d = 0; d < 8; d++) {
                const int tr = lr + cdy(d), tc = lc + cdx(d);
                const bool outside = tr < 0 || tr >= TH || tc < 0 || tc >= TW;
                const int pn = p + cdy(d) * FT::PW + cdx(d);
                const long y = i + (long)cdy(d) * W + cdx(d);
                // (an outlet's link is cut)
                id[d] = outside && T.smk[pn] && T.sfd[pn] == donor_code(d) && y != out ? a.exit_id[y] : -1;
            }
            unsigned long long e[8];
#pragma unroll
            for (int d = 0; d < 8; d++) e[d] = id[d] >= 0 ? a.ex_val[id[d]] : 0;
#pragma unroll
            for (int d = 0; d < 8; d++) in += e[d];
            at = lr * TW + lc;
        }
    }
#pragma unroll
    for (int q = 0; q < FT::PER; q++) {
        const int li = threadIdx.x + q * 256;
        const int lr = li / TW, lc = li % TW;
        const bool m = T.smk[fx_pad<TW>(lr, lc)];
        const long i = (long)(ty0 + lr) * W + tx0 + lc;
        T.x[li] = m ? x[q] : 0;
        T.J[li] = m ? fx_link(T, lr, lc, i == T.outlet[slot[q]]) : (uint16_t)FX_NONE;
    }
    __syncthreads();
    if (in) {
        for (int h = 0; at < (int)FX_EXIT && h < FT::NC; h++) {
            atomicAdd(&T.x[at], in);
            at = T.J[at];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < FT::PER; q++) {
        const int li = threadIdx.x + q * 256;
        const int lr = li / TW, lc = li % TW;
        const int r = ty0 + lr, col = tx0 + lc;
        if (r >= H || col >= W) continue;
        const long i = (long)r * W + col;
        if (!T.smk[fx_pad<TW>(lr, lc)]) {
            a.fa[i] = make_float2(0.f, 0.f);
            continue;
        }
        const unsigned long long s = T.x[li];
        if (i == T.outlet[slot[q]]) a.dsw[slot[q]].fx_outlet_sum = s;
        if (s >= FX_TAG) {
            const int k = atomicAdd(a.tag_count, 1);
            if (k < a.tag_cap) {
                a.tag_cell[k] = (int)i;
                a.tag_sum[k] = s;
            }
        } else {
            a.fa[i] = fx_value(s, T.shift[slot[q]]);
        }
    }
}

// exits listed, 0 if they are more than the list holds (the host then leaves the
// pass before its values are used)
__device__ __forceinline__ int fx_count(const int *count, int cap)
{
    const int n = *count;
    return n <= cap ? n : 0;
}

// parent of each exit in the exit forest; clears the counters of pass C
__global__ void k_fx_parent(const int *count, int cap, const int *ex_recv, const int *xroot, const int *exit_id, int *P,
                            int *tag_count, int *uncomputed)
{
    const int n = fx_count(count, cap);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *tag_count = 0;
        *uncomputed = 0;
    }
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int xr = xroot[ex_recv[k]];
        P[k] = xr >= 0 ? exit_id[xr] : -1;
    }
}

// one doubling round over the exit forest in two launches: snapshot, then add
__global__ void k_fx_gather(const int *count, int cap, const unsigned long long *val, const int *P,
                            unsigned long long *tv, int *tp, int *flag)
{
    const int n = fx_count(count, cap);
    if (blockIdx.x == 0 && threadIdx.x == 0) *flag = 0;   // raised by the scatter that follows
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int p = P[k];
        tv[k] = val[k];
        tp[k] = p >= 0 ? P[p] : -1;
    }
}

// Late rounds point many exits at the same few roots: the lanes of a wave
// with equal parents sit in runs, and each run's values are summed in the
// wave (a sum over the run's own lanes only, so every value counts once)
// and added by the run's first lane with one atomic.  Integer sums: the
// totals do not depend on the grouping.
__global__ void __launch_bounds__(256) k_fx_scatter(const int *count, int cap, unsigned long long *val, int *P,
                                                    const unsigned long long *tv, const int *tp, int *flag)
{
    const int lane = threadIdx.x & 63, n = fx_count(count, cap);
    bool more = false;
    // whole waves go round the loop together (the shuffles need every lane)
    for (int k0 = blockIdx.x * blockDim.x; k0 < n; k0 += gridDim.x * blockDim.x) {
        const int k = k0 + (int)threadIdx.x;
        int p = -1;
        unsigned long long v = 0;
        if (k < n) {
            p = P[k];
            if (p >= 0) {
                v = tv[k];
                const int q = tp[k];
                P[k] = q;
                more |= q >= 0;
            }
        }
        const int pprev = __shfl_up(p, 1, 64);
        const bool head = lane == 0 || pprev != p;
        const unsigned long long heads = __ballot(head);
        const unsigned long long above = lane == 63 ? 0ULL : heads & (~0ULL << (lane + 1));
        const int end = above ? __ffsll((long long)above) - 1 : 64;   // first lane of the next run
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const unsigned long long o = __shfl_down(v, off, 64);
            if (lane + off < end) v += o;
        }
        if (head && p >= 0) atomicAdd(&val[p], v);
    }
    if (__any(more) && lane == 0) *flag = 1;
}

// tagged cells: the cycle through the outlet (fa = w, never completed), or
// the path below the outlet (the outlet's sum added)
__global__ void k_fx_tags(const int *count, int cap, const int *tag_cell, const unsigned long long *tag_sum,
                          const uint8_t *demid, const DemScal *ds, const int *shift, const float *w, float2 *fa,
                          int *uncomputed)
{
    const int n = *count < cap ? *count : cap;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int i = tag_cell[k];
        const int s = demid ? (int)demid[i] : 0;
        const unsigned long long o = ds[s].fx_outlet_sum;
        if (o >= FX_TAG) {
            fa[i] = make_float2(w[i], 0.f);
            atomicAdd(uncomputed, 1);
        } else {
            fa[i] = fx_value(tag_sum[k] - FX_TAG + o, shift[s]);
        }
    }
}

static int fx_grid(long n)
{
    long g = (n + 255) / 256;
    if (g < 1) g = 1;
    if (g > 4096) g = 4096;
    return (int)g;
}

// fa as the runoff kernel left it.  Pass A keeps its sums there, and the
// engine writes only the cells that complete: those on a cycle through an
// outlet have to find fa = w.  (Bound by HBM; runs only before that engine.)
__global__ void __launch_bounds__(256) k_fx_undo(long N, const uint8_t *__restrict__ mask, const float *__restrict__ w,
                                                 float2 *__restrict__ fa)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x)
        fa[i] = make_float2(mask[i] ? w[i] : 0.f, 0.f);
}

// 0: done; 1: inputs the integer form cannot represent exactly (a negative
// or non-finite runoff weight, too many tagged cells, or a cycle that does not
// pass the outlet: directions from the caller, or an outlet moved after the
// direction phase) — the caller runs the dependency engine instead
int lem_fa32_sfd(lemhip_ctx *c, int *fallback)
{
    *fallback = 0;
    LEM_CHECK(c, hipMemcpyAsync(&c->hint[30], &c->scal->w_bad, sizeof(int), hipMemcpyDeviceToHost, c->s));
    LEM_TRY(lem_read_slots(c));
    if (c->hint[30]) { *fallback = 1; return LEMHIP_OK; }
    // per-slot shift: sums stay below 2^61 (the rounding adds at most N/2)
    for (int j = 0; j < c->nslot; j++) {
        const double tw = c->hdsc[j].totwater;
        int sh = 61;
        if (c->hdesc[j].w > 0) {
            if (!(tw >= 0.0) || tw > 1e300) { *fallback = 1; return LEMHIP_OK; }
            if (tw > 0.0) sh = 61 - (int)ceil(log2(tw * (1 + 1e-12)));
            if (sh > 1000) sh = 1000;
        }
        c->hfx_shift[j] = sh;
    }
    LEM_CHECK(c, hipMemcpyAsync(c->fx_shift, c->hfx_shift, sizeof(int) * c->nslot, hipMemcpyHostToDevice, c->s));
    const long N = c->N;
    FxArgs a;
    a.W = c->W;
    a.H = c->H;
    a.mask = c->mask;
    a.fd = c->fd;
    a.demid = c->demid;
    a.w = (const float *)c->w;
    a.ds = c->dsc;
    a.shift = c->fx_shift;
    a.nslot = c->nslot;
    a.exit_id = reinterpret_cast<int *>(c->scan_tmp);
    a.xroot = c->ws;
    unsigned long long *tv = reinterpret_cast<unsigned long long *>(c->z2);
    a.ex_val = tv + N / 2;
    a.ex_recv = c->cand;
    a.ex_count = &c->scal->nedges;
    a.ex_cap = (int)(N / 2);
    a.fa = reinterpret_cast<float2 *>(c->fa);
    a.tag_cell = c->fx_tag_cell;
    a.tag_sum = c->fx_tag_sum;
    a.tag_count = &c->scal->flag;
    a.tag_cap = (int)c->fx_tag_cap;
    a.dsw = c->dsc;
    auto leave = [&]() -> int {   // after pass A
        k_fx_undo<<<fx_grid(N), 256, 0, c->s>>>(N, a.mask, a.w, a.fa);
        LEM_LAUNCHED(c);
        *fallback = 1;
        return LEMHIP_OK;
    };
    constexpr int TW = 64, TH = 32;
    const long ntiles = (long)((c->W + TW - 1) / TW) * ((c->H + TH - 1) / TH);
    // A: in-tile sums, exits, in-tile roots of border cells
    LEM_CHECK(c, hipMemsetAsync(a.ex_count, 0, sizeof(int), c->s));
    k_fx_sums<TW, TH><<<ntiles, 256, 0, c->s>>>(a);
    LEM_LAUNCHED(c);
    // B: the exit forest.  The kernels take the number of exits from the device
    // and their grid from what it can be.
    const int ge = fx_grid(std::min(N, ntiles * FxTile<TW, TH>::NB));
    int *P = reinterpret_cast<int *>(c->sp0), *tp = reinterpret_cast<int *>(c->sp1);
    k_fx_parent<<<ge, 256, 0, c->s>>>(a.ex_count, a.ex_cap, a.ex_recv, a.xroot, a.exit_id, P, a.tag_count,
                                      &c->scal->fa_uncomputed);
    LEM_LAUNCHED(c);
    // rounds before the first host read: enough to double along a path that
    // crosses every tile row and column twice (a read leaves the device idle
    // for about 15 us, a round over a short list takes less); only a batch's
    // last round reports changes
    int batch = 2;
    while ((1 << batch) < 4 * ((c->W + TW - 1) / TW + (c->H + TH - 1) / TH)) batch++;
    for (int round = 0;; round += batch, batch = 2) {
        for (int q = 0; q < batch; q++) {
            k_fx_gather<<<ge, 256, 0, c->s>>>(a.ex_count, a.ex_cap, a.ex_val, P, tv, tp, &c->scal->nlabels);
            k_fx_scatter<<<ge, 256, 0, c->s>>>(a.ex_count, a.ex_cap, a.ex_val, P, tv, tp, &c->scal->nlabels);
        }
        LEM_LAUNCHED(c);
        LEM_CHECK(c, hipMemcpyAsync(c->hscal, c->scal, sizeof(LemScalars), hipMemcpyDeviceToHost, c->s));
        LEM_CHECK(c, hipStreamSynchronize(c->s));
        // the exit values and their snapshot share the 8-byte scratch of N
        // cells; exits are tile border cells (9% of a full tile), so only grids
        // of a few cells could have more
        if (c->hscal->nedges > a.ex_cap) return leave();
        if (!c->hscal->nlabels) break;
        if (round > 64) return leave();   // a cycle across tiles
    }
    // C: final sums, fa, tagged cells
    k_fx_final<TW, TH><<<ntiles, 256, 0, c->s>>>(a);
    LEM_LAUNCHED(c);
    k_fx_tags<<<64, 256, 0, c->s>>>(a.tag_count, a.tag_cap, a.tag_cell, a.tag_sum, c->demid, c->dsc, c->fx_shift,
                                    a.w, a.fa, &c->scal->fa_uncomputed);
    LEM_LAUNCHED(c);
    LEM_CHECK(c, hipMemcpyAsync(c->hscal, c->scal, sizeof(LemScalars), hipMemcpyDeviceToHost, c->s));
    LEM_CHECK(c, hipStreamSynchronize(c->s));
    if (c->hscal->flag > a.tag_cap) return leave();
    c->h_fa_unc = c->hscal->fa_uncomputed;
    c->dag_rounds_last = 0;
    return LEMHIP_OK;
}
