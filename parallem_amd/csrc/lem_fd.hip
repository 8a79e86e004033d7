// lem_fd.hip — flow direction phase (cuFlowDirection, routeflow.cu:686-975):
// D8/MFD directions, plateau routing, depression (sink) routing by watershed
// labels and minimax spill heights, the second direction pass on the raised
// surface, and the fd/SFD merge.
#include "lem_ctx.h"
#include <hipcub/hipcub.hpp>
#include <stddef.h>

// ------------------------------------------------------------------ helpers

// one atomic per wavefront: returns this lane's slot, or -1 if !pred
__device__ __forceinline__ int wave_append(int *counter, bool pred)
{
    unsigned long long b = __ballot(pred);
    if (b == 0) return -1;
    int lane = __lane_id();
    int leader = __ffsll((long long)b) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(counter, __popcll(b));
    base = __shfl(base, leader);
    return pred ? base + __popcll(b & ((1ULL << lane) - 1ULL)) : -1;
}

// one global atomic per workgroup (block size a multiple of 64, at most 1024);
// every thread of the block must call it
__device__ __forceinline__ int block_append(int *counter, bool pred, int *s_wave, int *s_base)
{
    unsigned long long b = __ballot(pred);
    int tid = threadIdx.y * blockDim.x + threadIdx.x;
    int lane = tid & 63;
    int wave = tid >> 6;
    int nwaves = (blockDim.x * blockDim.y) >> 6;
    if (lane == 0) s_wave[wave] = __popcll(b);
    __syncthreads();
    if (tid == 0) {
        int tot = 0;
        for (int w = 0; w < nwaves; w++) {
            int cnt = s_wave[w];
            s_wave[w] = tot;
            tot += cnt;
        }
        *s_base = tot ? atomicAdd(counter, tot) : 0;
    }
    __syncthreads();
    int pos = *s_base + s_wave[wave] + __popcll(b & ((1ULL << lane) - 1ULL));
    __syncthreads();
    return pred ? pos : -1;
}

// n_mine items per thread appended to a global list with one atomic per block;
// returns this thread's first index
__device__ __forceinline__ int block_append_n(int *counter, int n_mine, int *s_wave, int *s_base)
{
    int tid = threadIdx.y * blockDim.x + threadIdx.x;
    int lane = tid & 63;
    int wave = tid >> 6;
    int nwaves = (blockDim.x * blockDim.y) >> 6;
    int x = n_mine;   // inclusive scan within the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    if (tid == 0) {
        int tot = 0;
        for (int w = 0; w < nwaves; w++) {
            int cnt = s_wave[w];
            s_wave[w] = tot;
            tot += cnt;
        }
        *s_base = tot ? atomicAdd(counter, tot) : 0;
    }
    __syncthreads();
    int pos = *s_base + s_wave[wave] + x - n_mine;
    __syncthreads();
    return pos;
}

// Stream compaction in chunks of 256 * ITEMS elements (1-D blocks of 256):
// one global atomic per chunk instead of one per 256 elements, since many
// workgroups adding to one counter serialise.  Output order is a permutation
// within each chunk.
#define COMPACT_ITEMS 16
template <int ITEMS, class Pred, class Emit>
__device__ __forceinline__ void compact_chunks(long n, int *count, int *s_wave, int *s_base, Pred pred, Emit emit)
{
    const long CH = 256L * ITEMS;
    for (long c0 = blockIdx.x * CH; c0 < n; c0 += (long)gridDim.x * CH) {
        unsigned keep = 0;
        int mine = 0;
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            long i = c0 + j * 256 + threadIdx.x;
            bool k = i < n && pred(i);
            keep |= (unsigned)k << j;
            mine += k;
        }
        int pos = block_append_n(count, mine, s_wave, s_base);
#pragma unroll
        for (int j = 0; j < ITEMS; j++)
            if ((keep >> j) & 1u) emit(c0 + j * 256 + threadIdx.x, pos++);
    }
}

// The same keeping the input order: the chunk is read row by row (256
// consecutive elements, coalesced); one atomic reserves the chunk's output
// range, then each row's kept elements take their ranks from a block-wide
// scan of that row.
template <int ITEMS, class Pred, class Emit>
__device__ __forceinline__ void compact_chunks_ordered(long n, int *count, int *s_wave, int *s_base, Pred pred,
                                                       Emit emit)
{
    __shared__ int s_row[ITEMS][4];
    const long CH = 256L * ITEMS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (long c0 = blockIdx.x * CH; c0 < n; c0 += (long)gridDim.x * CH) {
        unsigned keep = 0;
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            long i = c0 + j * 256 + threadIdx.x;
            bool k = i < n && pred(i);
            keep |= (unsigned)k << j;
            unsigned long long b = __ballot(k);
            if (lane == 0) s_row[j][wave] = __popcll(b);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int tot = 0;
            for (int j = 0; j < ITEMS; j++)
                for (int w = 0; w < 4; w++) {
                    int c = s_row[j][w];
                    s_row[j][w] = tot;
                    tot += c;
                }
            *s_base = tot ? atomicAdd(count, tot) : 0;
        }
        __syncthreads();
        const int base = *s_base;
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            bool k = (keep >> j) & 1u;
            unsigned long long b = __ballot(k);
            if (k) emit(c0 + j * 256 + threadIdx.x, base + s_row[j][wave] + __popcll(b & ((1ULL << lane) - 1ULL)));
        }
        __syncthreads();
    }
}

static inline int grid_chunks(long n, int cap = 8192, int items = COMPACT_ITEMS)
{
    long g = (n + 256L * items - 1) / (256L * items);
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return (int)g;
}

template <typename T>
__device__ __forceinline__ T block_reduce_sum(T v, T *sh)
{
    int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] += sh[t + s];
        __syncthreads();
    }
    T r = sh[0];
    __syncthreads();
    return r;
}

// ----------------------------------------------------------------- lowest

// routeflow.cu:739-741: the outlet is lowered below the lowest cell after the
// directions were computed on the unadjusted surface (one thread per slot)
__global__ void k_slots_outlet_adjust(double *dem, uint8_t *fd, const DemDesc *dd, int ns, DemScal *ds)
{
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ns || dd[j].w == 0) return;
    double lowest = ord_dec(ds[j].lowest_enc);
    ds[j].lowest = lowest;
    if (lowest < dem[ds[j].outlet]) dem[ds[j].outlet] = lowest - 0.0001;
    fd[ds[j].outlet] = 16;   // routeflow.cu:953: WEST
}

// per-slot counter adds from a block: LDS histogram over slots, then one atomic per slot touched
__device__ __forceinline__ void slot_hist_flush(int *hist, DemScal *ds, int off, int ns)
{
    __syncthreads();
    for (int j = threadIdx.x; j < ns; j += blockDim.x)
        if (hist[j]) atomicAdd(reinterpret_cast<int *>(reinterpret_cast<char *>(&ds[j]) + off), hist[j]);
}

// ---------------------------------------------------------------- FlowDirs

// newflow.cu:49-174.  One thread per cell; a wave covers 64 consecutive cells
// of a row so the centre row and both neighbour rows are read coalesced.
// Slopes take new values only for downhill neighbours (sticky: Slopes keep the first pass's values); pass 2
// passes slopes == nullptr.  Cells without a downhill neighbour are appended
// to the plateau candidate list (the cells whose initial distance is 2e7).
// A 64 x 4 block covers nsub (at most four) 64 x 16 tiles: each tile's
// surface plus a one-cell ring is staged in LDS with every load in flight at
// once, then each thread evaluates four rows from LDS.  The block appends its
// candidates with one atomic at the end (appends from many blocks to one
// counter serialise).  Off-grid ring cells hold NaN: every comparison with it
// is false, so such a neighbour is neither downhill, up nor flat, exactly as
// a skipped one.
template <typename TS>
__global__ void __launch_bounds__(256) k_flowdirs(int W, int H, int nsub, int cell_size, const double *__restrict__ z,
                                                  const uint8_t *__restrict__ mask, TS *__restrict__ slopes,
                                                  long plane, uint8_t *__restrict__ fd, uint8_t *__restrict__ SFD,
                                                  uint8_t *__restrict__ eqb, float *__restrict__ sp,
                                                  int *__restrict__ cand, int *__restrict__ ncand)
{
    constexpr int RW = 66, RH = 18, RN = RW * RH, PER = (RN + 255) / 256;
    __shared__ double zs[RN];
    __shared__ int s_wave[4];
    __shared__ int s_base;
    const int tid = threadIdx.y * 64 + threadIdx.x;
    const int x0 = blockIdx.x * 64;
    const int icol = x0 + threadIdx.x;
    unsigned cand_rows = 0;   // bit 4 * sub + rg: the cell of row group rg of tile sub is a plateau candidate
    for (int sub = 0; sub < nsub; sub++) {
        const int y0 = (blockIdx.y * nsub + sub) * 16;
        if (y0 >= H) break;
        double v[PER];
#pragma unroll
        for (int q = 0; q < PER; q++) {
            int k = tid + q * 256;
            int gy = y0 - 1 + k / RW, gx = x0 - 1 + k % RW;
            v[q] = lm_nan();
            if (k < RN && gy >= 0 && gy < H && gx >= 0 && gx < W) v[q] = z[(long)gy * W + gx];
        }
        uint32_t mk[4];   // 32-bit: byte registers would be packed, with a wait per load
#pragma unroll
        for (int rg = 0; rg < 4; rg++) {
            int irow = y0 + rg * 4 + threadIdx.y, icol = x0 + threadIdx.x;
            mk[rg] = (icol < W && irow < H) ? mask[(long)irow * W + icol] : 0;
        }
        __syncthreads();   // the previous tile's reads are done
#pragma unroll
        for (int q = 0; q < PER; q++) {
            int k = tid + q * 256;
            if (k < RN) zs[k] = v[q];
        }
        __syncthreads();
#pragma unroll 1
        for (int rg = 0; rg < 4; rg++) {
            int lr = rg * 4 + threadIdx.y;
            int irow = y0 + lr;
            bool inside = icol < W && irow < H;
            long self = (long)irow * W + icol;
            bool active = inside && mk[rg];
            int aspect = 0, aspectsfd = 0;
            unsigned eq = 0;
            if (active) {
                // Every Slopes plane of the cell is rewritten, keeping the old value
                // where the neighbour is not downhill: whole cache lines are written
                // instead of lines with holes in them.  The old values are loaded
                // first and merged after the scan.
                TS sv[8];
                if (slopes) {
#pragma unroll
                    for (int d = 0; d < 8; d++) sv[d] = slopes[d * plane + self];
                }
                const int c0 = (lr + 1) * RW + (threadIdx.x + 1);
                double zc = zs[c0];
                double smax = 0.0;
                int up = 0, flat = 0;
                unsigned down = 0;
                TS nv[8];
#pragma unroll
                for (int d = 0; d < 8; d++) {
                    float dc = (d & 1) ? 1.41f : 1.0f;
                    float den = (float)cell_size * dc;
                    double zn = zs[c0 + kDY[d] * RW + kDX[d]];
                    double stemp = (zc - zn) / (double)den;
                    nv[d] = (TS)stemp;
                    if ((zc > zn) && (zn != -9999)) {
                        down |= 1u << d;
                        if (stemp > smax) { smax = stemp; aspectsfd = kCODE[d]; }
                        aspect += kCODE[d];
                    }
                    if (zc < zn) up++;
                    if (zc == zn) { flat++; eq |= 1u << d; }
                }
                if (slopes) {
#pragma unroll
                    for (int d = 0; d < 8; d++) slopes[d * plane + self] = ((down >> d) & 1u) ? nv[d] : sv[d];
                }
                if (up > 7) { aspect = 0; aspectsfd = 0; }
                if ((flat + up) > 7 && up <= 7) { aspect = 0; aspectsfd = 0; }
                if ((flat < 8) && (flat + up > 7)) { aspect = 0; aspectsfd = 0; }
            }
            const bool is_cand = active && aspect == 0 && aspectsfd == 0;
            if (inside) {
                fd[self] = (uint8_t)aspect;
                SFD[self] = (uint8_t)aspectsfd;
                eqb[self] = (uint8_t)eq;
                // candidates start at 2e7 (newflow.cu:252), the rest keep 0 and never change
                sp[self] = is_cand ? 20000000.0f : 0.0f;
            }
            if (is_cand) cand_rows |= 1u << (sub * 4 + rg);
        }
    }
    // one append per block for its candidates (their order is not needed)
    int mine = __popc(cand_rows);
    int base = block_append_n(ncand, mine, s_wave, &s_base);
    while (cand_rows) {
        const int b = __ffs(cand_rows) - 1;
        cand_rows &= cand_rows - 1;
        cand[base++] = (int)((long)((blockIdx.y * nsub + (b >> 2)) * 16 + (b & 3) * 4 + threadIdx.y) * W + icol);
    }
}

// ------------------------------------------------------------ plateaus
//
// route_plateausMFD (newflow.cu:264-350) in synchronous rounds: in round
// r a candidate reads its equal-height neighbours' round r-1 distances; each
// strict improvement in the scan (order N..NW) marks that slope and takes its
// direction.  The rounds are temporally blocked: one launch advances K rounds
// for a tile of PTW x PTH cells, loading the tile plus a K-cell halo into LDS
// and recomputing the halo redundantly; after round k only cells at least k
// cells from the halo's outer edge are current, so after K rounds the tile
// itself is exact.  A cell can change in round r only if an equal-height
// neighbour changed in round r-1, so a tile needs the next launch only when a
// cell within K cells of it changed in the last round of this launch (K <=
// tile width and height: in it or in one of its 8 neighbour tiles); tiles
// without candidates never change.

// Launch bookkeeping: launch L visits list L % 3 (count cnt[L % 3]); a tile
// still moving at its end queues itself and its neighbours with candidates in
// list (L+1) % 3, each once (stamp[tile] holds the last launch it was queued
// for), and launch L clears cnt[(L+2) % 3], last read by the publish step of
// launch L-1.
struct PlatCtl {
    int cnt[3];
    int pad0[29];
    int last_change;   // last round (absolute number) in which any cell changed
    int ncand;         // plateau candidates (mask cells without a downhill neighbour)
    int cut;           // some sink label has no path to label 0 (pass 2: known after the surface was raised)
    int pad1[29];
};

// everything a pass starts from but its distances
__global__ void k_plat_init(int ntiles, int *tile_has, int *tver, PlatCtl *ctl)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < ntiles) {
        tile_has[t] = 0;
        tver[t] = -2;   // buffer 0, written before any launch
    }
    if (t < 3) ctl->cnt[t] = 0;
    if (t == 3) ctl->last_change = 0;
    if (t == 4) ctl->ncand = 0;
}

// the tiles with candidates (their number is read on the device, so the host
// does not wait for it)
__global__ void k_sp_seed(int W, const int *cand, const PlatCtl *ctl, int ntx, int *tile_has)
{
    const int n = ctl->ncand;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int i = cand[k];
        const int t = ((i / W) / PTH) * ntx + (i % W) / PTW;
        if (tile_has[t] == 0) tile_has[t] = 1;
    }
}

// A candidate with an equal-height neighbour at distance 0 (not a
// candidate, or off the grid, where the plateau rounds read 0) takes its
// distance in the first round; every other cell changes in round r only if
// an equal-height neighbour changed in round r-1, i.e. it lies within r-1
// cells of such a seed.  The first launch's K rounds (K <= tile height) can
// therefore change only tiles in the 3x3 tile neighbourhood of a seed's
// tile: those tiles (with candidates) are marked 3, the first list.
__global__ void k_sp_seedmark(int W, int H, const int *cand, const PlatCtl *ctl, const float *sp, const uint8_t *eqb,
                              int ntx, int nty, int *tile_has)
{
    const int n = ctl->ncand;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int i = cand[k];
        const int y = i / W, x = i % W;
        const unsigned e = eqb[i];
        bool seed = false;
#pragma unroll
        for (int d = 0; d < 8; d++) {
            const int yy = y + cdy(d), xx = x + cdx(d);
            if ((e >> d) & 1u) seed |= yy < 0 || yy >= H || xx < 0 || xx >= W || sp[(long)yy * W + xx] == 0.0f;
        }
        if (!seed) continue;
        const int ty = y / PTH, tx = x / PTW;
        for (int dy = -1; dy <= 1; dy++)
            for (int dx = -1; dx <= 1; dx++) {
                const int t2y = ty + dy, t2x = tx + dx;
                if (t2y < 0 || t2y >= nty || t2x < 0 || t2x >= ntx) continue;
                const int t2 = t2y * ntx + t2x;
                if (tile_has[t2] != 0) tile_has[t2] = 3;
            }
    }
}

__global__ void k_plat_first_list(int ntiles, const int *tile_has, int *list, PlatCtl *ctl, int slot)
{
    __shared__ int s_wave[4];
    __shared__ int s_base;
    for (int t0 = blockIdx.x * blockDim.x; t0 < ntiles; t0 += gridDim.x * blockDim.x) {
        int t = t0 + threadIdx.x;
        bool have = t < ntiles && tile_has[t] == 3;
        int at = block_append(&ctl->cnt[slot], have, s_wave, &s_base);
        if (have) list[at] = t;
    }
}

// threads per plateau workgroup: a launch near the end of the pass (16 rounds)
// visits a few tiles, so its rounds are spread over all the waves a workgroup
// can have (512^2 DEM, pass on the filled surface: 0.19 ms against 0.22 with
// 512 threads); with many tiles moving 512 threads hold more tiles at once
// (4096^2: 1.97 ms, 2.22 with 1024)
#define PLAT_NT(K) ((K) == 16 ? 1024 : 512)

// Distances live in two buffers per tile: tver[tile] = 2 * (launch that last
// wrote the tile) + (buffer it wrote).  A launch reads every tile from the
// buffer holding its state as of the previous launch and a visited tile
// writes the other one, so no launch reads what another visit of the same
// launch writes, and no copy-back is needed.
__device__ __forceinline__ int plat_buf_as_of(int tv, int launch)
{
    int b = tv & 1;
    return (tv >> 1) == launch ? 1 - b : b;
}

// Appends a workgroup's queued tiles to the next launch's list with one
// atomic (called by every thread of the workgroup, after a barrier).
#define PLAT_QCAP 1024
__device__ __forceinline__ void plat_flush(int *qbuf, int *qn, int *next, int *count)
{
    __shared__ int base;
    const int cnt = *qn;
    if (threadIdx.x == 0) base = atomicAdd(count, cnt);
    __syncthreads();
    for (int k = threadIdx.x; k < cnt; k += blockDim.x) next[base + k] = qbuf[k];
    __syncthreads();
    if (threadIdx.x == 0) *qn = 0;
    __syncthreads();
}

// MARKS: the pass records slope marks (the first pass, on the dem; the pass
// on the raised surface keeps only directions and distances)
//
// A visit is bound by the latency of its K rounds: 12.4 of a tail visit's
// 17 us when every cell was evaluated in every round.  In a round only the
// cells next to a change of the round before can change: a front a few cells
// wide.  The region is therefore cut into 8 x 8 blocks, one wave evaluates a
// block at a time, and a block is evaluated only when it or the adjacent edge
// of a neighbour block changed in the last round (a front of any orientation
// meets about a quarter of the blocks); a wave reads the stamps of all its
// blocks at once, a cell its neighbours, and one flag tells whether the last
// round changed anything.  5.6 us of 11 for 8 rounds, and the first launch over
// a 4096^2 DEM 245 -> 182 us; the pass 3.05 -> 1.97 ms, on 1201^2 0.93 -> 0.57.
// Blocks are dealt to the waves so that a row or column of them falls on
// different waves; the LDS pitch is an odd number of 8-cell groups, so a
// block's rows lie in different banks.
template <int K, typename TS, bool MARKS>
__global__ void __launch_bounds__(PLAT_NT(K), K == 16 ? 4 : 6) k_plat_block(int W, int H, int launch, int r0,
                                                    int kn, const int *__restrict__ act, int *__restrict__ next, float *__restrict__ sp0,
                                                    float *__restrict__ sp1, int *__restrict__ tver,
                                                    const uint8_t *__restrict__ eqb,
                                                    uint8_t *__restrict__ fd, uint8_t *__restrict__ SFD,
                                                    TS *__restrict__ slopes, long plane,
                                                    const int *__restrict__ tile_has, int *__restrict__ tstamp,
                                                    PlatCtl *ctl)
{
    constexpr int RW = PTW + 2 * K, RH = PTH + 2 * K, RN = RW * RH, NI = PTW * PTH;
    constexpr int NT = PLAT_NT(K), PER = (RN + NT - 1) / NT, PERI = (NI + NT - 1) / NT;
    constexpr int NBX = RW / 8, NBY = RH / 8, NB = NBX * NBY, NW = NT / 64, BPW = (NB + NW - 1) / NW;
    constexpr int P = (NBX & 1) ? RW : RW + 8, LN = P * RH;   // LDS pitch
    constexpr int G = P + 1;                                  // guard: every cell's neighbours can be read
    constexpr int SX = NBX + 2;                               // pitch of the block stamps (a ring of unused ones)
    static_assert(RW % 8 == 0 && RH % 8 == 0 && (NW & (NW - 1)) == 0, "8 x 8 blocks dealt to the waves");
    __shared__ uint32_t bufA[LN + 2 * G], bufB[LN + 2 * G];   // distances as bits: none is negative, so they order as unsigned
    // equal-height bits, and above them the distance from the region's edge: a
    // cell is current after round k when that is at least k (0: never changes)
    __shared__ uint16_t E[LN];
    __shared__ uint8_t code[NI], marks[NI];
    __shared__ uint8_t stamp[2][SX * (NBY + 2)];   // by round parity: the last round the block is due in
    __shared__ int s_any[K + 1];   // some cell changed in that round
    __shared__ int last;
    __shared__ int s_qmask;   // 3x3 tiles within kn cells of a cell that changed in round K
    __shared__ int s_buf[9], s_has[9];
    __shared__ int qbuf[PLAT_QCAP];   // tiles queued for the next launch, not yet appended
    __shared__ int qn;
    int wg_last = 0;                  // thread 0: the last round with a change in this workgroup's visits
    uint32_t *const A = bufA + G, *const B = bufB + G;
    if (threadIdx.x == 0) qn = 0;
    const int n = ctl->cnt[launch % 3];
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->cnt[(launch + 2) % 3] = 0;
    const int ntx = (W + PTW - 1) / PTW, nty = (H + PTH - 1) / PTH;
    // the cell of a block this lane evaluates, and (lanes 0-8) the neighbour
    // block it stamps with the cells of a block that are adjacent to it
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int ly = lane >> 3, lx = lane & 7;
    const int wy = lane / 3 - 1, wx = lane % 3 - 1;
    unsigned long long adj = ~0ULL;
    if (wy < 0) adj &= 0xFFULL;
    if (wy > 0) adj &= 0xFFULL << 56;
    if (wx < 0) adj &= 0x0101010101010101ULL;
    if (wx > 0) adj &= 0x8080808080808080ULL;
    if (lane >= 9) adj = 0;
    // block `lane` of this wave's (lanes below BPW): its stamp
    const int myb = lane * NW + ((wave - 3 * lane) & (NW - 1));
    const int mys = lane < BPW && myb < NB ? (myb / NBX + 1) * SX + myb % NBX + 1 : -1;
    // the next visit's tile is read during this one (the first together with
    // the count: the grid never exceeds the list's capacity, and an entry
    // past the count is never used)
    int tile_next = act[blockIdx.x];
    for (int q0 = blockIdx.x; q0 < n; q0 += gridDim.x) {
        const int tile = tile_next;
        tile_next = q0 + (int)gridDim.x < n ? act[q0 + gridDim.x] : 0;
        const int tx0 = (tile % ntx) * PTW, ty0 = (tile / ntx) * PTH;
        __syncthreads();
        if (threadIdx.x == 0) { last = 0; s_qmask = 0; }
        if (threadIdx.x < 2 * SX * (NBY + 2)) stamp[0][threadIdx.x] = 0;   // both parities
        if (threadIdx.x <= K) s_any[threadIdx.x] = 0;
        // load the region from both distance buffers, and in the same wait
        // which buffer holds each of the 3x3 tiles as of the last launch: the
        // region's loads do not wait for that choice (a visit of the first
        // launches spends most of its time waiting on its loads)
        float v0[PER], v1[PER];
        uint32_t e[PER];   // 32-bit: byte registers would be packed, with a wait per load
        int part[PER];   // 3x3 tile of the region cell, -1 off the grid
#pragma unroll
        for (int q = 0; q < PER; q++) {
            int idx = threadIdx.x + q * NT;
            int gy = ty0 - K + idx / RW, gx = tx0 - K + idx % RW;
            v0[q] = 0.f;
            v1[q] = 0.f;
            e[q] = 0;
            part[q] = -1;
            if (idx < RN && gy >= 0 && gy < H && gx >= 0 && gx < W) {
                long i = (long)gy * W + gx;
                int ny = gy < ty0 ? 0 : (gy >= ty0 + PTH ? 2 : 1), nx = gx < tx0 ? 0 : (gx >= tx0 + PTW ? 2 : 1);
                part[q] = ny * 3 + nx;
                v0[q] = sp0[i];
                v1[q] = sp1[i];
                e[q] = eqb[i];
            }
        }
        if (threadIdx.x < 9) {
            int ty = tile / ntx + (int)threadIdx.x / 3 - 1, tx = tile % ntx + (int)threadIdx.x % 3 - 1;
            const bool in = ty >= 0 && ty < nty && tx >= 0 && tx < ntx;
            const int tv = in ? tver[ty * ntx + tx] : 0;
            s_has[threadIdx.x] = in ? tile_has[ty * ntx + tx] : 0;
            s_buf[threadIdx.x] = in ? plat_buf_as_of(tv, launch) : 0;
        }
        __syncthreads();
        // both LDS buffers hold every cell, so cells that cannot change (no
        // candidate, or no equal-height neighbour) are never rewritten
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int idx = threadIdx.x + q * NT;
            const float v = part[q] < 0 ? 0.f : (s_buf[part[q]] ? v1[q] : v0[q]);
            if (idx < RN) {
                const int rr = idx / RW, cc = idx % RW, li = rr * P + cc;
                const int dy = rr < RH - 1 - rr ? rr : RH - 1 - rr, dx = cc < RW - 1 - cc ? cc : RW - 1 - cc;
                A[li] = __float_as_uint(v);
                B[li] = __float_as_uint(v);
                E[li] = v != 0.f && e[q] != 0 ? (uint16_t)(e[q] | ((dy < dx ? dy : dx) << 8)) : 0;
            }
        }
#pragma unroll
        for (int q = 0; q < PERI; q++) {
            int li = threadIdx.x + q * NT;
            if (li < NI) { code[li] = 0; marks[li] = 0; }
        }
        __syncthreads();
        uint32_t *cur = A, *nxt = B;
        int moved = 0;   // last round in which one of this thread's tile cells changed
        unsigned qm = 0;  // 3x3 tiles within kn cells of this thread's cells that changed in round K
        // A round in which no cell of its window changes leaves every later
        // round unchanged too (round k+1 reads only round k values of a window
        // that contains its own), so the launch stops there.  A block not due
        // in round k did not change in round k-1, so both buffers hold it.
        for (int k = 1; k <= K; k++) {
            // the blocks due of this wave, one bit each, and whether the last
            // round changed anything: one LDS wait
            unsigned due = (1u << BPW) - 1;
            if (k > 1) {
                const int st = mys >= 0 ? stamp[k & 1][mys] : 0;
                const int any = s_any[k - 1];
                if (!any) break;
                due = (unsigned)__ballot(st == k);
            }
            bool changed = false;
            while (due) {
                const int j = __ffs(due) - 1;
                due &= due - 1;
                const int blk = j * NW + ((wave - 3 * j) & (NW - 1)), by = blk / NBX, bx = blk - by * NBX;
                if (NB % NW && blk >= NB) continue;
                // every read of the cell in flight at once (lanes whose cell
                // is not current read within the guard and discard)
                const int b = (by * 8 + ly) * P + bx * 8 + lx;
                const uint32_t ee = E[b], md0 = cur[b];
                uint32_t c[8];
#pragma unroll
                for (int d = 0; d < 8; d++) c[d] = cur[b + cdy(d) * P + cdx(d)];
                const int dep = (int)(ee >> 8);
                // the scan N..NW takes the smallest distance below the cell's
                // own, the first direction that has it; directions without an
                // equal-height neighbour count as beyond every distance
                uint32_t m = ~0u;
#pragma unroll
                for (int d = 0; d < 8; d++) {
                    const float dis = __uint_as_float(c[d]) + ((d & 1) ? 1.41f : 1.0f);
                    c[d] = __float_as_uint(dis) | (uint32_t)((int)(~ee << (31 - d)) >> 31);
                    m = c[d] < m ? c[d] : m;
                }
                const bool on = dep >= k, ch = on && m < md0;
                if (on) nxt[b] = ch ? m : md0;
                const unsigned long long M = __ballot(ch);
                if (!M) continue;
                changed = true;
                if (M & adj) stamp[(k + 1) & 1][(by + 1) * SX + bx + 1 + wy * SX + wx] = (uint8_t)(k + 1);
                if (ch && dep >= K) {   // a changed cell of the tile
                    unsigned cd = 0;
#pragma unroll
                    for (int d = 7; d >= 0; d--) cd = c[d] == m ? (1u << ((d + 6) & 7)) : cd;   // fd code of direction d
                    const int ty = by * 8 + ly - K, tx = bx * 8 + lx - K;
                    code[ty * PTW + tx] = (uint8_t)cd;
                    if (MARKS) {
                        uint32_t md = md0;
                        unsigned mk = 0;
#pragma unroll
                        for (int d = 0; d < 8; d++) {
                            const bool take = c[d] < md;
                            md = take ? c[d] : md;
                            mk |= take ? (1u << d) : 0u;
                        }
                        marks[ty * PTW + tx] |= (uint8_t)mk;
                    }
                    moved = k;
                    if (k == K) {
                        const unsigned rows = 2u | (ty < kn ? 1u : 0u) | (ty >= PTH - kn ? 4u : 0u);
                        const unsigned cols = 2u | (tx < kn ? 1u : 0u) | (tx >= PTW - kn ? 4u : 0u);
#pragma unroll
                        for (int ny = 0; ny < 3; ny++)
                            if ((rows >> ny) & 1u) qm |= cols << (3 * ny);
                    }
                }
            }
            if (changed) s_any[k] = 1;
            __syncthreads();
            uint32_t *t = cur; cur = nxt; nxt = t;
        }
        if (moved) atomicMax(&last, moved);
        if (qm) atomicOr(&s_qmask, (int)qm);
        __syncthreads();
        // still moving at the end of the launch: this tile and the neighbours
        // within kn cells of a cell that changed in the last round go on (a
        // cell changing in round K + j lies within j cells of one that changed
        // in round K, and the next launch takes at most kn rounds), gathered in LDS and appended to the next list with one
        // atomic per full buffer (workgroups adding to one counter serialise).
        // Before the write-back: the wait for the atomic's returned value
        // would otherwise also wait for those stores
        if (threadIdx.x < 9 && ((s_qmask >> threadIdx.x) & 1)) {
            int ty = tile / ntx + (int)threadIdx.x / 3 - 1, tx = tile % ntx + (int)threadIdx.x % 3 - 1;
            if (ty >= 0 && ty < nty && tx >= 0 && tx < ntx) {
                const int t2 = ty * ntx + tx;
                if (s_has[threadIdx.x] && atomicExch(&tstamp[t2], launch + 1) != launch + 1) qbuf[atomicAdd(&qn, 1)] = t2;
            }
        }
        // write back the tile: distances (into its other buffer), directions of
        // changed cells, slope marks (pass 1 only)
        float *sp_out = s_buf[4] ? sp0 : sp1;
#pragma unroll
        for (int q = 0; q < PERI; q++) {
            int li = threadIdx.x + q * NT;
            int gy = ty0 + li / PTW, gx = tx0 + li % PTW;
            if (li >= NI || gy >= H || gx >= W) continue;
            long i = (long)gy * W + gx;
            sp_out[i] = __uint_as_float(cur[(li / PTW + K) * P + (li % PTW + K)]);
            uint8_t cd = code[li];
            if (cd) { fd[i] = cd; SFD[i] = cd; }
            if (MARKS && marks[li]) {
                unsigned mk = marks[li];
#pragma unroll
                for (int d = 0; d < 8; d++)
                    if ((mk >> d) & 1) slopes[d * plane + i] = (TS)0.0001;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            tver[tile] = (launch << 1) | (s_buf[4] ? 0 : 1);
            if (last > 0 && r0 + last > wg_last) wg_last = r0 + last;
        }
        __syncthreads();
        if (qn > PLAT_QCAP - 9) plat_flush(qbuf, &qn, next, &ctl->cnt[(launch + 1) % 3]);
    }
    __syncthreads();
    if (qn > 0) plat_flush(qbuf, &qn, next, &ctl->cnt[(launch + 1) % 3]);
    if (threadIdx.x == 0 && wg_last > 0) atomicMax(&ctl->last_change, wg_last);
}

// the sinks per DEM, and the counts and flag of the label phase
__global__ void k_slots_sinks_init(int ns, DemScal *ds, LemScalars *sc)
{
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < ns) ds[j].sinks_pass1 = 0;
    if (j == 0) {
        sc->sinks_pass1 = 0;
        sc->ncand = 0;
        sc->flag = 0;
    }
}

__global__ void __launch_bounds__(256) k_count_sinks(const int *cand, int n, const uint8_t *SFD,
                                                     const uint8_t *demid, int ns, DemScal *ds, int *total)
{
    __shared__ int hist[LEM_MAX_SLOTS + 1];
    int mine = 0;
    for (int j = threadIdx.x; j < ns; j += blockDim.x) hist[j] = 0;
    __syncthreads();
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        long i = cand[k];
        if (SFD[i] == 0) {
            atomicAdd(&hist[slot_of(demid, i)], 1);
            mine = 1;
        }
    }
    slot_hist_flush(hist, ds, (int)offsetof(DemScal, sinks_pass1), ns);
    if (mine) *total = 1;   // some DEM has sinks
}

// ------------------------------------------------ watershed labels

// DEM-local border of init_watershedMFD (newflow.cu:371): last column, first
// and last row of the cell's own DEM
// A cell of a DEM lies in its last column, first row or last row exactly when
// its east, north or south neighbour is outside the DEM's rectangle: off the
// grid, or in another DEM's rectangle or none (rectangles are convex).  The
// three slot ids are read at once instead of the DEM's rectangle after the
// cell's own id.
__device__ __forceinline__ bool dem_border(int W, int H, int r, int c, long i, const uint8_t *demid)
{
    if (demid) {
        const uint8_t me = demid[i];
        const uint8_t e = c + 1 < W ? demid[i + 1] : DEM_NONE;
        const uint8_t n = r > 0 ? demid[i - W] : DEM_NONE;
        const uint8_t s = r + 1 < H ? demid[i + W] : DEM_NONE;
        return e != me || n != me || s != me;
    }
    return (c == W - 1) || (r == 0) || (r == H - 1);
}

// sink flag: mask, not on the DEM border, SFD == 0 (newflow.cu:363-378)
// Row/column grids (grid2d): cell coordinates without a division per cell.
__global__ void k_sink_flags(int W, int H, const uint8_t *mask, const uint8_t *SFD, const uint8_t *demid,
                             const DemDesc *dd, int *flag)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= W) return;
    for (int r = blockIdx.y; r < H; r += gridDim.y) {
        const long i = (long)r * W + c;
        const uint8_t m = mask[i], s = SFD[i];   // both loads in flight
        flag[i] = (m && s == 0 && !dem_border(W, H, r, c, i, demid)) ? 1 : 0;
    }
}

// init_watershedMFD with labels = 1 + rank of the sink cell in atlas row-major order
__global__ void k_init_ws(int W, int H, const uint8_t *mask, const uint8_t *SFD, const int *prefix,
                          const uint8_t *demid, const DemDesc *dd, int *ws, uint8_t *labdem, int *nlab)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= W) return;
    for (int r = blockIdx.y; r < H; r += gridDim.y) {
        const long i = (long)r * W + c;
        const uint8_t m = mask[i], s = SFD[i];   // loads in flight together
        const int sl = slot_of(demid, i);
        int v;
        if (!m) v = 0;
        else if (dem_border(W, H, r, c, i, demid)) v = 0;
        else if (s == 0) {
            v = prefix[i] + 1;
            labdem[v] = (uint8_t)sl;
        } else {
            int d = code_dir(s);
            v = -((r + kDY[d]) * W + (c + kDX[d]) + 1);
        }
        ws[i] = v;
        if (r == H - 1 && c == W - 1) *nlab = prefix[i] + (v > 0 ? 1 : 0);
    }
}

// init_watershed_sinkMFD (newflow.cu:430-460): SFD==0 cells adopt the largest
// label of an equal-height neighbour; iterated to the fixed point (the
// component maximum, independent of the update order).  SFD==0 cells are a
// subset of the pass-1 plateau candidates.
__global__ void k_sink_merge(int W, int H, const int *cand, const int *count, const uint8_t *SFD, const double *z,
                             int *ws, int *flag)
{
    const int n = *count;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        long self = cand[k];
        if (SFD[self] != 0) continue;
        int irow = (int)(self / W), icol = (int)(self % W);
        double zc = z[self];
        int cur = ws[self], best = cur;
        for (int d = 0; d < 8; d++) {
            int cx = icol + kDX[d], cy = irow + kDY[d];
            if (cx >= 0 && cx < W && cy >= 0 && cy < H) {
                long nb = (long)cy * W + cx;
                if (z[nb] == zc) {
                    int v = ws[nb];
                    if (v > best) best = v;
                }
            }
        }
        if (best > cur) { ws[self] = best; *flag = 1; }
    }
}

// Only sinks with an equal-height neighbour can change in the merge above;
// they are collected once (the equal-height bits come from the FlowDirs pass on
// the same surface) and the merge iterates over them alone.
__global__ void __launch_bounds__(256) k_merge_list(const int *cand, int n, const uint8_t *SFD, const uint8_t *eqb,
                                                    int *list, int *count)
{
    __shared__ int s_wave[4];
    __shared__ int s_base;
    for (int k0 = blockIdx.x * blockDim.x; k0 < n; k0 += gridDim.x * blockDim.x) {
        int k = k0 + threadIdx.x;
        int i = k < n ? cand[k] : 0;
        bool keep = k < n && SFD[i] == 0 && eqb[i] != 0;
        int at = block_append(count, keep, s_wave, &s_base);
        if (keep) list[at] = i;
    }
}

// identify_watershedMFD (newflow.cu:469-487): pointer jumping, LINKS links;
// in-place reads of already-jumped targets only shorten chains
// (clears the flag of the walks and the count of the edge list)
template <int LINKS>
__global__ void k_jump(long N, const uint8_t *mask, int *ws, int *flag, int *nedges)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *flag = *nedges = 0;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) {
        const uint8_t m = mask[i];   // loads in flight together
        int v = ws[i];
        if (v >= 0 || !m) continue;
        for (int q = 0; q < LINKS && v < 0; q++) v = ws[-v - 1];
        ws[i] = v;
    }
}

// The rest in one launch: every cell still pointing walks to its label, and
// leaves its progress behind every eight links, so the walks behind it skip
// ahead.  (Walks that left only their label took 1.10 ms on a smooth 2000x1500
// DEM, paths of up to some 3000 cells; a list of the cells still pointing and
// launches over it until none was left cost two host reads and nine launches
// more: 0.12 ms of a 512^2 DEM's step.)  A walk ends after `limit` links and
// says so: the cells downstream of a long path may not have started yet, and
// then a winding valley is walked link by link (see WS_JUMPS).
__global__ void k_jump_walk(long N, const uint8_t *mask, int *ws, int limit, int *more)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) {
        int v = ws[i];
        if (v >= 0 || !mask[i]) continue;
        int hops = 0;
        do {
            v = __hip_atomic_load(&ws[-v - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (v < 0 && (++hops & 7) == 0) __hip_atomic_store(&ws[i], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } while (v < 0 && hops < limit);
        if (v < 0) *more = 1;
        ws[i] = v;
    }
}

// ------------------------------------------------------ edges, spill

#define HASH_EMPTY 0xFFFFFFFFFFFFFFFFULL

__device__ __forceinline__ unsigned long long mix64(unsigned long long k)
{
    k ^= k >> 33; k *= 0xff51afd7ed558ccdULL; k ^= k >> 33; k *= 0xc4ceb9fe1a85ec53ULL; k ^= k >> 33;
    return k;
}

// identify_watershed_boundary_write_backMFD (newflow.cu:787-877) without the
// fixed-size table: every mask cell c and in-grid neighbour n with different
// labels and z_c >= z_n contributes edge {ws_c, ws_n} at height z_c, and the
// edge list keeps the minimum per unordered pair (order-free, exact).  The
// cells of a block share most of their basin pairs (a boundary runs through
// many cells): pairs are first merged in an LDS table (minimum weight per
// pair), and each block appends its distinct pairs to a list with one atomic;
// pairs that find no LDS slot are appended one by one.  Blocks of 64 x 16
// cells with a 1024-entry table (16 KB) keep eight blocks resident per
// compute unit.  Each neighbour pair is looked at once, from its upper or left
// cell (with the weights either cell would give it; eight directions per cell
// before), by threads that take four rows with every load in flight together:
// 4096^2 310 -> 189 us, 1201^2 43 -> 27, 512^2 26 -> 15.  The list is then
// sorted by pair and reduced to the minimum weight per pair.  Keys pack
// (lo << B) | hi with B bits per label.  The count may exceed the capacity:
// the caller then grows the list and runs again.
#define EDGE_LDS 1024
#define EDGE_RG 4   // rows per thread: blocks of 64 x (4 * EDGE_RG) cells
__global__ void __launch_bounds__(256) k_edges_emit(int W, int H, const uint8_t *__restrict__ mask,
                                                    const int *__restrict__ ws, const double *__restrict__ z,
                                                    const uint8_t *__restrict__ demid, unsigned long long *keys,
                                                    unsigned long long *vals, long cap, int *count, int B,
                                                    const int *unfinished)
{
    if (*unfinished) return;   // some cell has no label yet: the host runs this again
    __shared__ unsigned long long lk[EDGE_LDS], lv[EDGE_LDS];
    __shared__ int s_wave[4];
    __shared__ int s_base;
    const unsigned long long NONE = ~0ULL;   // no height encodes to it
    const int tid = threadIdx.y * blockDim.x + threadIdx.x;
    for (int q = tid; q < EDGE_LDS; q += 256) { lk[q] = HASH_EMPTY; lv[q] = HASH_EMPTY; }
    __syncthreads();
    const int x = blockIdx.x * 64 + threadIdx.x, y0 = (blockIdx.y * 4 + threadIdx.y) * EDGE_RG;
    if (x < W) {
        // rows y0 .. y0 + EDGE_RG of this column and the two beside it, every
        // load in flight together; D holds the DEM (off the grid: none that a
        // cell could have) and bit 9 the mask
        int L[EDGE_RG + 1][3];
        double Z[EDGE_RG + 1][3];
        uint32_t D[EDGE_RG + 1][3], M[EDGE_RG + 1][3];
#pragma unroll
        for (int r = 0; r <= EDGE_RG; r++)
#pragma unroll
            for (int q = r ? 0 : 1; q < 3; q++) {
                const int cx = x + q - 1, cy = y0 + r;
                const bool in = cx >= 0 && cx < W && cy < H;
                const long n = in ? (long)cy * W + cx : 0;
                L[r][q] = ws[n];
                Z[r][q] = z[n];
                M[r][q] = in ? mask[n] : 0;
                D[r][q] = in ? (demid ? demid[n] : 0) : 0x100;
            }
#pragma unroll
        for (int r = 0; r <= EDGE_RG; r++)
#pragma unroll
            for (int q = r ? 0 : 1; q < 3; q++) D[r][q] |= M[r][q] ? 0x200 : 0;
#pragma unroll
        for (int r = 0; r < EDGE_RG; r++) {
            const int me = L[r][1];
            const double zc = Z[r][1];
            const unsigned long long ec = ord_enc(zc);
            // the four pairs: east, south-west, south, south-east; pairs with
            // the same label are one
            int oth[4];
            unsigned long long w[4];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const int pr = p ? r + 1 : r, pq = p ? p - 1 : 2;
                const double zn = Z[pr][pq];
                const bool pair = L[pr][pq] != me && ((D[pr][pq] ^ D[r][1]) & 0x1FF) == 0;
                unsigned long long v = NONE;
                if (pair && (D[r][1] & 0x200) && zc >= zn) v = ec;
                const unsigned long long en = ord_enc(zn);
                if (pair && (D[pr][pq] & 0x200) && zn >= zc && en < v) v = en;
                oth[p] = L[pr][pq];
                w[p] = v;
#pragma unroll
                for (int q = 0; q < p; q++)
                    if (oth[q] == oth[p] && w[q] != NONE && w[p] != NONE) {
                        w[q] = w[p] < w[q] ? w[p] : w[q];
                        w[p] = NONE;
                    }
            }
#pragma unroll
            for (int p = 0; p < 4; p++) {
                if (w[p] == NONE) continue;
                const int other = oth[p];
                unsigned long long lo = (unsigned)(me < other ? me : other), hi = (unsigned)(me < other ? other : me);
                unsigned long long key = (lo << B) | hi;
                unsigned h = (unsigned)(mix64(key) & (EDGE_LDS - 1));
                bool done = false;
                for (int t = 0; t < 16 && !done; t++) {
                    unsigned long long prev = atomicCAS(&lk[h], HASH_EMPTY, key);
                    if (prev == HASH_EMPTY || prev == key) { atomicMin(&lv[h], w[p]); done = true; }
                    h = (h + 1) & (EDGE_LDS - 1);
                }
                if (!done) {
                    int at = atomicAdd(count, 1);
                    if (at < cap) { keys[at] = key; vals[at] = w[p]; }
                }
            }
        }
    }
    __syncthreads();
    constexpr int PERT = EDGE_LDS / 256;
    int mine = 0;
#pragma unroll
    for (int j = 0; j < PERT; j++) mine += lk[tid * PERT + j] != HASH_EMPTY;
    int pos = block_append_n(count, mine, s_wave, &s_base);
#pragma unroll
    for (int j = 0; j < PERT; j++) {
        unsigned long long key = lk[tid * PERT + j];
        if (key == HASH_EMPTY) continue;
        if (pos < cap) { keys[pos] = key; vals[pos] = lv[tid * PERT + j]; }
        pos++;
    }
}

// unique pairs (sorted) to the edge list; label flags as in the compaction
__global__ void k_edges_decode(const int *cnt, const unsigned long long *ukeys, const unsigned long long *uw, int B,
                               uint32_t *elo, uint32_t *ehi, unsigned long long *ew, uint8_t *seen,
                               const uint8_t *labdem, DemScal *ds)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= *cnt) return;
    unsigned long long key = ukeys[k];
    uint32_t lo = (uint32_t)(key >> B), hi = (uint32_t)(key & ((1ULL << B) - 1));
    elo[k] = lo;
    ehi[k] = hi;
    ew[k] = uw[k];
    if (!seen[lo]) seen[lo] = 1;
    if (!seen[hi]) seen[hi] = 1;
    if (lo == 0 && !ds[labdem[hi]].zero_seen) ds[labdem[hi]].zero_seen = 1;
}

// nothing to flood: every slot's sink count (newflow.cu:1045: data->sinkcount, the
// distinct labels in the edge set, counted by k_bv_init) is 0
__global__ void k_slots_sinkcount_init(int ns, DemScal *ds)
{
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ns) return;
    ds[j].sinkcount = 0;
    ds[j].zero_seen = 0;
}

// label 0 counts as one of a slot's labels when the slot has an edge to it;
// a slot without sinks skipped flooding and reports its sink count
__global__ void k_slots_sinkcount_fin(const DemDesc *dd, int ns, DemScal *ds)
{
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= ns || dd[j].w == 0) return;
    if (ds[j].sinks_pass1 == 0) ds[j].sinkcount = 0;
    else ds[j].sinkcount += ds[j].zero_seen;
}

// spill heights and label marks; the DEMs' sink counts, the flag of the
// walks and the cut-off flag
__global__ void k_minimax_init(long n, unsigned long long *r, uint8_t *seen, int ns, DemScal *ds, int *flag, int *cut)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < ns) {
        ds[j].sinkcount = 0;
        ds[j].zero_seen = 0;
    }
    if (j == 0) *flag = *cut = 0;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        r[i] = (i == 0) ? ord_enc(-lm_inf()) : ord_enc(lm_inf());
        seen[i] = 0;
    }
}

// Bottleneck distance to label 0 over the basin graph:
// r[b] = min over edges (b,c) of max(w_bc, r[c]), r[0] = -inf.  This is the
// value the reference's Kruskal/union-find pass assigns (routeflow.cu:529-572):
// a basin is raised to the height at which it first joins label 0 in
// ascending-weight order.  Relaxation in any order reaches the same fixed point.
__global__ void k_minimax_relax(int ne, const uint32_t *elo, const uint32_t *ehi, const unsigned long long *ew,
                                unsigned long long *r, int *flag)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ne) return;
    uint32_t a = elo[k], b = ehi[k];
    unsigned long long w = ew[k];
    unsigned long long ra = r[a], rb = r[b];
    unsigned long long ca = w > rb ? w : rb;
    unsigned long long cb = w > ra ? w : ra;
    if (ca < ra) { atomicMin(&r[a], ca); *flag = 1; }
    if (cb < rb) { atomicMin(&r[b], cb); *flag = 1; }
}

// ---- spill heights by Borůvka phases
//
// The bottleneck distance above (the relaxation's fixed point) equals the
// heaviest edge on the minimum spanning tree's path from label 0, with edges
// ordered by encoded weight and then by position in the label-sorted list (a
// strict total order, so the tree is unique).  Borůvka builds that tree in
// phases: every component takes its lightest outgoing edge, and the chosen
// edges join components.  In the tree of components the phases form (each
// component a child of the one it joins, that edge weighing what the
// component chose), the heaviest edge between two leaves equals the
// heaviest edge on the spanning tree's path between them (V. King, "A
// simpler minimum spanning tree verification algorithm", Algorithmica 18,
// 1997).  So a label v that joins label 0's component in phase p gets
//     r(v) = max(-inf, the weights v's components chose in phases 1..p,
//                the weights label 0's components chose in phases 1..p),
// both running maxima, one per label and one for label 0.  Edges of weight
// +inf or above (encoded) lower nothing in the relaxation and are left out;
// a label that never joins keeps +inf (the cut-off fallback below takes
// those).  About log2(labels) phases instead of one relaxation pass per
// link of the longest bottleneck path.
//
// Per phase (bw/be: the chosen weight and edge per component, double-buffered
// by phase parity; nxt: the component each root joins):
// st[0], st[1]: label 0's running maximum and its component (st[2], st[3] in
// odd phases)
// (the labels of the edge set are counted per DEM on the way, ns = 0: they have
// been; heights: the spill heights an earlier start of the phases left, reset)
__global__ void __launch_bounds__(256) k_bv_init(long n, uint32_t *comp, unsigned long long *mv,
                                                 unsigned long long *bw0, unsigned long long *bw1, uint32_t *be0,
                                                 uint32_t *be1, unsigned long long *st, const uint8_t *seen,
                                                 const uint8_t *labdem, int ns, DemScal *ds,
                                                 unsigned long long *heights)
{
    __shared__ int hist[LEM_MAX_SLOTS + 1];
    for (int j = threadIdx.x; j < ns; j += blockDim.x) hist[j] = 0;
    __syncthreads();
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        if (heights) heights[i] = ord_enc(i == 0 ? -lm_inf() : lm_inf());
        comp[i] = (uint32_t)i;
        mv[i] = 0ULL;
        bw0[i] = bw1[i] = ~0ULL;
        be0[i] = be1[i] = ~0u;
        if (i == 0) st[0] = st[1] = 0ULL;
        else if (ns && seen[i]) atomicAdd(&hist[labdem[i]], 1);
    }
    slot_hist_flush(hist, ds, (int)offsetof(DemScal, sinkcount), ns);
}

// the lightest outgoing weight of each component.  The edge list is sorted
// by (lo, hi), so the lanes of a wave whose edges leave one component on
// the lo side sit in runs: each run's weights are reduced in the wave
// (a minimum over edges of one component, in any grouping) and only the
// run's first lane updates the component, instead of one atomic per lane
// on the same address; the same for runs on the hi side.
__global__ void __launch_bounds__(256) k_bv_min_w(const int *cnt, const uint32_t *__restrict__ lo,
                                                  const uint32_t *__restrict__ hi,
                                                  const unsigned long long *__restrict__ w,
                                                  const uint32_t *__restrict__ comp, unsigned long long *bw)
{
    const unsigned long long INF = ord_enc(lm_inf());
    const int k = blockIdx.x * blockDim.x + threadIdx.x, ne = *cnt;
    const int lane = threadIdx.x & 63;
    bool live = false;
    unsigned long long wk = ~0ULL;
    uint32_t ca = ~0u, cb = ~0u;
    if (k < ne) {
        wk = w[k];
        ca = comp[lo[k]];
        cb = comp[hi[k]];
        live = ca != cb && wk < INF;
    }
    // lanes without an edge to count carry a key no component has; the hi
    // side's components repeat in runs too once components have merged
    uint32_t key = live ? ca : ~0u, key2 = live ? cb : ~0u;
    unsigned long long v = live ? wk : ~0ULL, v2 = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long ov = __shfl_down(v, off, 64), ov2 = __shfl_down(v2, off, 64);
        const uint32_t okey = __shfl_down(key, off, 64), okey2 = __shfl_down(key2, off, 64);
        if (lane + off < 64 && okey == key && ov < v) v = ov;
        if (lane + off < 64 && okey2 == key2 && ov2 < v2) v2 = ov2;
    }
    // every lane takes part in the shuffles (a shuffle under a branch would
    // read the inactive lane 0 as 0, component 0's key)
    const uint32_t prev = __shfl_up(key, 1, 64), prev2 = __shfl_up(key2, 1, 64);
    const bool head = lane == 0 || prev != key;
    const bool head2 = lane == 0 || prev2 != key2;
    if (live && head && v < bw[ca]) atomicMin(&bw[ca], v);
    if (live && head2 && v2 < bw[cb]) atomicMin(&bw[cb], v2);
}

// the first edge of that weight
__global__ void k_bv_min_e(const int *cnt, const uint32_t *__restrict__ lo, const uint32_t *__restrict__ hi,
                           const unsigned long long *__restrict__ w, const uint32_t *__restrict__ comp,
                           const unsigned long long *__restrict__ bw, uint32_t *be)
{
    const unsigned long long INF = ord_enc(lm_inf());
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= *cnt) return;
    const unsigned long long wk = w[k];
    const uint32_t ca = comp[lo[k]], cb = comp[hi[k]];
    if (ca == cb || wk >= INF) return;
    if (wk == bw[ca]) atomicMin(&be[ca], (uint32_t)k);
    if (wk == bw[cb]) atomicMin(&be[cb], (uint32_t)k);
}

// A component with a chosen edge points at the component across it (every
// other label at itself).  Two components that chose the same edge would
// point at each other (under a strict order no longer cycle forms): the
// smaller is the root.  The edge counter of this phase's compaction is cleared.
__global__ void k_bv_hook(long n, const uint32_t *__restrict__ lo, const uint32_t *__restrict__ hi,
                          const uint32_t *__restrict__ comp, const uint32_t *__restrict__ be, uint32_t *nxt, int *kept)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        if (i == 0) *kept = 0;
        const uint32_t e = be[i];
        uint32_t t = (uint32_t)i;
        if (e != ~0u) {
            const uint32_t a = comp[lo[e]], b = comp[hi[e]];
            const uint32_t o = a == (uint32_t)i ? b : a;
            if (be[o] != e || o < (uint32_t)i) t = o;
        }
        nxt[i] = t;
    }
}

// pointer jumping towards the roots, launched only once a walk below gave up
__global__ void k_bv_jump(long n, uint32_t *nxt)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const uint32_t t = nxt[i];
        const uint32_t tt = nxt[t];
        if (tt != t) nxt[i] = tt;
    }
}

// The root of component c's joined component: the pointers form trees whose
// roots point at themselves (the only cycles Borůvka's choices make under a
// strict order are pairs, and k_bv_hook turns those into roots).  Most paths
// have a few links (pointer jumping launched before the walks cost more than it
// saved: 0.22 instead of 0.19 ms for the phases on 1201^2).  In a longer path,
// a row of basins with rising sills, each walker leaves its progress at its own
// component every eight links, so walkers behind it skip ahead.  A path can
// have as many links as there are labels, and label 0's walk runs in every
// block before any other has shortened its path, so a walk of more than
// BV_WALK_MAX links raises the flag instead: the host then starts the phases
// again with jumps before the walks (260 K basins joining along one path: a
// step of 4.7 ms, 390 to 630 with walks to the end).
#define BV_WALK_MAX 512
__device__ __forceinline__ uint32_t bv_root(uint32_t *nxt, uint32_t c, int *over)
{
    uint32_t x = nxt[c];
    for (int h = 0; h < 8; h++) {
        const uint32_t y = nxt[x];
        if (y == x) return x;
        x = y;
    }
    for (int h = 0; h < BV_WALK_MAX; h++) {
        if ((h & 7) == 0) __hip_atomic_store(&nxt[c], x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t y = __hip_atomic_load(&nxt[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (y == x) return x;
        x = y;
    }
    *over = 1;
    return x;
}

// every label: its running maximum, its new component, and its spill height
// if that component is label 0's (whose own maximum and root each block finds
// by itself: st as of this phase, stn for the next); the other parity's
// entries are reset for the next phase (each label its own)
__global__ void k_bv_labels(long n, uint32_t *comp, const unsigned long long *__restrict__ bw,
                            const uint32_t *__restrict__ be, uint32_t *nxt,
                            unsigned long long *mv, unsigned long long *r, const unsigned long long *st,
                            unsigned long long *stn, unsigned long long *bwn, uint32_t *ben, int *over)
{
    const unsigned long long INF = ord_enc(lm_inf()), NEG = ord_enc(-lm_inf());
    __shared__ unsigned long long s_m0;
    __shared__ uint32_t s_root0;
    if (threadIdx.x == 0) {
        const uint32_t c0 = (uint32_t)st[1];
        unsigned long long m = st[0];
        if (be[c0] != ~0u && bw[c0] > m) m = bw[c0];
        s_m0 = m;
        s_root0 = bv_root(nxt, c0, over);
        if (blockIdx.x == 0) {
            stn[0] = m;
            stn[1] = s_root0;
        }
    }
    __syncthreads();
    const unsigned long long m0 = s_m0;
    const uint32_t root0 = s_root0;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        const uint32_t c = comp[i];
        unsigned long long m = mv[i];
        if (be[c] != ~0u && bw[c] > m) m = bw[c];
        mv[i] = m;
        const uint32_t nc = bv_root(nxt, c, over);
        comp[i] = nc;
        bwn[i] = ~0ULL;
        ben[i] = ~0u;
        if (i != 0 && nc == root0 && r[i] == INF) {
            unsigned long long v = m > m0 ? m : m0;
            r[i] = v > NEG ? v : NEG;
        }
    }
}

// edges between different components, in order (chunks of 4 rows on short
// lists: with 16, the 27 K edges of a 512^2 DEM ran in 7 workgroups, 14.6 us a
// phase; on long ones fewer workgroups add to the one counter)
template <int ITEMS>
__global__ void __launch_bounds__(256) k_bv_keep(const int *cnt, const uint32_t *elo, const uint32_t *ehi,
                                                 const unsigned long long *ew, const uint32_t *comp, uint32_t *lo2,
                                                 uint32_t *hi2, unsigned long long *w2, int *count)
{
    __shared__ int s_wave[4];
    __shared__ int s_base;
    const unsigned long long INF = ord_enc(lm_inf());
    compact_chunks_ordered<ITEMS>(
        *cnt, count, s_wave, &s_base, [&](long k) { return ew[k] < INF && comp[elo[k]] != comp[ehi[k]]; },
        [&](long k, int at) { lo2[at] = elo[k]; hi2[at] = ehi[k]; w2[at] = ew[k]; });
}

// Basins with no path to label 0 (only possible when NaN heights cut them
// off): the reference's union-find never marks them done, merges them in
// ascending order and leaves every member with the height of the component's
// last merge, i.e. the largest edge of the component's minimum spanning tree.
// That equals max over v of the bottleneck distance from any one member, so
// the component's smallest label seeds a second relaxation and the component
// takes the maximum.
__global__ void k_fb_unreached(int ne, const uint32_t *elo, const uint32_t *ehi, const unsigned long long *r, int *flag)
{
    const unsigned long long INF = ord_enc(lm_inf());
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < ne && (r[elo[k]] == INF || r[ehi[k]] == INF)) *flag = 1;
}

__global__ void k_fb_comp_init(long n, uint32_t *comp, unsigned long long *cmax)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        comp[i] = (uint32_t)i;
        cmax[i] = 0ULL;
    }
}

__global__ void k_fb_comp_relax(int ne, const uint32_t *elo, const uint32_t *ehi, const unsigned long long *r,
                                uint32_t *comp, int *flag)
{
    const unsigned long long INF = ord_enc(lm_inf());
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ne) return;
    uint32_t a = elo[k], b = ehi[k];
    if (r[a] != INF || r[b] != INF) return;
    uint32_t ca = comp[a], cb = comp[b];
    if (ca < cb) { atomicMin(&comp[b], ca); *flag = 1; }
    else if (cb < ca) { atomicMin(&comp[a], cb); *flag = 1; }
}

// seeds: the smallest label of each cut-off component; other cut-off labels
// restart from +inf in a separate array (cmax doubles as that array)
__global__ void k_fb_seed(long n, const unsigned long long *r, const uint32_t *comp, const uint8_t *seen,
                          unsigned long long *r2)
{
    const unsigned long long INF = ord_enc(lm_inf());
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        r2[i] = (r[i] == INF && seen[i] && comp[i] == (uint32_t)i) ? ord_enc(-lm_inf()) : INF;
}

__global__ void k_fb_max(long n, const unsigned long long *r, const uint32_t *comp, const uint8_t *seen,
                         const unsigned long long *r2, unsigned long long *out)
{
    const unsigned long long INF = ord_enc(lm_inf());
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        if (r[i] == INF && seen[i] && r2[i] != INF && r2[i] != ord_enc(-lm_inf())) atomicMax(&out[comp[i]], r2[i]);
}

__global__ void k_fb_apply(long n, unsigned long long *r, const uint32_t *comp, const uint8_t *seen,
                           const unsigned long long *out)
{
    const unsigned long long INF = ord_enc(lm_inf());
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        if (r[i] == INF && seen[i] && out[comp[i]] != 0ULL) r[i] = out[comp[i]];
}

// raise_watershedMFD (newflow.cu:879-894) into a copy of the surface; label 0
// and labels without a path keep raise = 0 as in the reference's zeroed array
__global__ void k_raise(long N, const uint8_t *mask, const int *ws, const unsigned long long *r,
                        const double *z, const uint8_t *demid, const DemScal *ds, double *z2)
{
    const unsigned long long INF = ord_enc(lm_inf());
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) {
        double v = z[i];
        const uint8_t m = mask[i];   // the cell's own loads in flight together
        const int lab = ws[i];
        const int sl = slot_of(demid, i);
        // floodingDriver only runs for a DEM with sinks left (routeflow.cu:913)
        if (m && ds[sl].sinks_pass1 > 0) {
            unsigned long long e = r[lab];
            double rs = (lab == 0 || e == INF) ? 0.0 : ord_dec(e);
            if (v < rs) v = rs;
        }
        z2[i] = v;
    }
}

// routeflow.cu:938-953
__global__ void k_merge(long N, int flowtype, const uint8_t *mask, uint8_t *fd, const uint8_t *SFD)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) {
        uint8_t f = fd[i];
        if (flowtype == 0) f = SFD[i];
        else if (f == 0 && mask[i]) f = SFD[i];
        fd[i] = f;
    }
}

// ------------------------------------------------------------ host side

static int grid1d(long n, int block = 256, int cap = 8192)
{
    long g = (n + block - 1) / block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (int)g;
}

// 256-thread blocks over the columns, a row per block row (rows beyond the
// grid's height are taken in strides)
static dim3 grid2d(int W, int H)
{
    return dim3((unsigned)((W + 255) / 256), (unsigned)(H < 32768 ? (H > 0 ? H : 1) : 32768));
}

static int read_scalars(lemhip_ctx *c)
{
    LEM_CHECK(c, hipMemcpyAsync(c->hscal, c->scal, sizeof(LemScalars), hipMemcpyDeviceToHost, c->s));
    LEM_CHECK(c, hipStreamSynchronize(c->s));
    return LEMHIP_OK;
}

static int clear_flag(lemhip_ctx *c)
{
    LEM_CHECK(c, hipMemsetAsync(&c->scal->flag, 0, sizeof(int), c->s));
    return LEMHIP_OK;
}

static int read_flag(lemhip_ctx *c, int *v)
{
    LEM_CHECK(c, hipMemcpyAsync(&c->hscal->flag, &c->scal->flag, sizeof(int), hipMemcpyDeviceToHost, c->s));
    LEM_CHECK(c, hipStreamSynchronize(c->s));
    *v = c->hscal->flag;
    return LEMHIP_OK;
}

// workgroups the chip holds of each plateau kernel a context uses: fewer than
// 16 rounds per launch and 16, without and with slope marks
template <typename TS>
static int plat_grids(lemhip_ctx *c)
{
    const void *f[2][2] = {{(const void *)k_plat_block<8, TS, false>, (const void *)k_plat_block<8, TS, true>},
                           {(const void *)k_plat_block<16, TS, false>, (const void *)k_plat_block<16, TS, true>}};
    for (int q = 0; q < 2; q++)
        for (int m = 0; m < 2; m++) {
            int bpc = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, f[q][m], q ? PLAT_NT(16) : PLAT_NT(8), 0) != hipSuccess || bpc < 1) bpc = 1;
            c->plat_grid[q][m] = bpc * c->ncu;
        }
    return LEMHIP_OK;
}

// FlowDirs + plateau routing on surface zs; slopes == nullptr for pass 2.
// Leaves the candidate list in c->cand and its length in *ncand_out; returns
// the number of rounds that changed something in *rounds, all read after the
// first launches.  cut (pass 2): set, and the pass left, when labels turn out
// to be cut off from label 0.
template <typename TS>
static int directions_and_plateaus(lemhip_ctx *c, const double *zs, TS *slopes, int *ncand_out, int *rounds,
                                   bool *cut = nullptr)
{
    long N = c->N;
    int W = c->W, H = c->H;
    uint8_t *eqb = c->dmask;   // equal-height neighbour bits; the accumulation passes reuse the buffer later
    const int ntx = (W + PTW - 1) / PTW, nty = (H + PTH - 1) / PTH, ntiles = ntx * nty;
    int *tile_has = c->pl_tiles, *tstamp = c->pl_tiles + ntiles, *tver = c->pl_tiles + 5 * (long)ntiles;
    int *L[3] = {c->pl_tiles + 2 * (long)ntiles, c->pl_tiles + 3 * (long)ntiles, c->pl_tiles + 4 * (long)ntiles};
    PlatCtl *ctl = reinterpret_cast<PlatCtl *>(c->pl_ctl);
    float *sp_in = c->sp0, *sp_out = c->sp1;
    int launch = c->pl_launch;
    if (launch > (1 << 29)) {  // tile stamps hold launch numbers: restart them well before they wrap
        LEM_CHECK(c, hipMemsetAsync(tstamp, 0, ntiles * sizeof(int), c->s));
        launch = 0;
    }
    k_plat_init<<<(ntiles + 255) / 256, 256, 0, c->s>>>(ntiles, tile_has, tver, ctl);
    dim3 blk(64, 4);
    // four tiles per block once that makes two blocks for each compute unit
    // (one tile throughout: 0.42 instead of 0.38 ms for both passes on 4096^2),
    // else one (four: 57 instead of 34 us on 512^2, 75 instead of 62 on 1201^2)
    const int nsub = (long)((W + 63) / 64) * ((H + 63) / 64) >= 2L * c->ncu ? 4 : 1;
    dim3 grd((W + 63) / 64, (H + 16 * nsub - 1) / (16 * nsub));
    prof_begin(c, PROF_FLOWDIRS);
    k_flowdirs<TS><<<grd, blk, 0, c->s>>>(W, H, nsub, (int)c->p.cellsize, zs, c->mask, slopes, c->NP, c->fd, c->SFD, eqb,
                                          sp_in, c->cand, &ctl->ncand);
    prof_end(c, PROF_FLOWDIRS);
    LEM_LAUNCHED(c);
    prof_begin(c, PROF_PLATEAU);
    // about a tenth of the cells or fewer are candidates
    const int gc = grid1d(N / 16, 256, 8192);
    k_sp_seed<<<gc, 256, 0, c->s>>>(W, c->cand, ctl, ntx, tile_has);
    k_sp_seedmark<<<gc, 256, 0, c->s>>>(W, H, c->cand, ctl, sp_in, eqb, ntx, nty, tile_has);
    k_plat_first_list<<<grid1d(ntiles, 256, 1024), 256, 0, c->s>>>(ntiles, tile_has, L[launch % 3], ctl, launch % 3);
    LEM_LAUNCHED(c);
    // Eight rounds per launch while many tiles move (with 16 throughout, the
    // wider halo makes the pass 2.9 instead of 2.0 ms on 4096^2), 16 once they
    // are no more than the compute units, where a launch costs about 9 us
    // whatever it does (8 throughout: 2.17 ms on 4096^2, 0.68 instead of 0.57
    // on 1201^2).  The last launch of a
    // batch queues the tiles a launch of 16 rounds could reach.
    const bool widen = c->plat_k == 8;
    int K = widen && ntiles <= c->ncu ? 16 : c->plat_k;
    int G[2] = {c->plat_grid[0][slopes ? 1 : 0], c->plat_grid[1][slopes ? 1 : 0]};   // of K < 16 and K = 16
    if (!G[0]) {
        LEM_TRY(plat_grids<TS>(c));
        for (int q = 0; q < 2; q++) G[q] = c->plat_grid[q][slopes ? 1 : 0];
    }
    int r = 0;  // rounds done in this pass
    int n = 0;
    long guard = 0;
    // launches between host checks (an empty launch costs less than a read);
    // the first pass seldom has a flat to drain
    for (int batch = slopes ? 4 : 128 / K;; batch = 128 / K) {
        prof_begin(c, PROF_PLAT_K);
        for (int q = 0; q < batch; q++) {
            const int *a_cur = L[launch % 3];
            int *a_next = L[(launch + 1) % 3];
            const int grid = G[K == 16] < ntiles ? G[K == 16] : ntiles;
            const int kn = q == batch - 1 && widen ? 16 : K;
            switch (K) {
#define PLAT_LAUNCH(K)                                                                                           \
    if (slopes)                                                                                                  \
        k_plat_block<K, TS, true><<<grid, PLAT_NT(K), 0, c->s>>>(W, H, launch, r, kn, a_cur, a_next, sp_in, sp_out, tver, \
                                                              eqb, c->fd, c->SFD, slopes, c->NP, tile_has, tstamp, ctl); \
    else                                                                                                         \
        k_plat_block<K, TS, false><<<grid, PLAT_NT(K), 0, c->s>>>(W, H, launch, r, kn, a_cur, a_next, sp_in, sp_out, tver, \
                                                               eqb, c->fd, c->SFD, slopes, c->NP, tile_has, tstamp, ctl)
            case 4: PLAT_LAUNCH(4); break;
            case 16: PLAT_LAUNCH(16); break;
            default: PLAT_LAUNCH(8); break;
#undef PLAT_LAUNCH
            }
            ++launch;
            r += K;
        }
        prof_end(c, PROF_PLAT_K, batch);
        LEM_LAUNCHED(c);
        PlatCtl *h = reinterpret_cast<PlatCtl *>(c->hint + 64);
        LEM_CHECK(c, hipMemcpyAsync(h, ctl, sizeof(PlatCtl), hipMemcpyDeviceToHost, c->s));
        LEM_CHECK(c, hipStreamSynchronize(c->s));
        n = h->ncand;
        *ncand_out = n;
        *rounds = h->last_change;
        if (cut) {
            *cut = h->cut != 0;
            if (*cut) break;   // the surface has to be raised again: this pass is repeated
        }
        const int moving = h->cnt[launch % 3];
        if (moving == 0) break;   // nothing queued for the next launch
        if (widen && moving <= c->ncu) K = 16;
        // every launch with a moving tile changes at least one cell, and a
        // cell's distance only decreases through a finite set of path lengths
        if (++guard > (long)n + 2) { c->err = "plateau routing did not converge"; return LEMHIP_E_NOT_CONVERGED; }
    }
    c->pl_launch = launch;
    prof_end(c, PROF_PLATEAU, *rounds + 1);
    return LEMHIP_OK;
}

static int ensure_hash(lemhip_ctx *c, long want)
{
    long cap = 1024;
    while (cap < want) cap <<= 1;
    if (cap <= c->hcap) return LEMHIP_OK;
    if (c->hkeys) { (void)hipFree(c->hkeys); (void)hipFree(c->hvals); (void)hipFree(c->elo); (void)hipFree(c->ehi); (void)hipFree(c->ew); }
    for (int q = 0; q < 2; q++) {
        if (c->elo2[q]) { (void)hipFree(c->elo2[q]); (void)hipFree(c->ehi2[q]); (void)hipFree(c->ew2[q]); }
        c->elo2[q] = c->ehi2[q] = nullptr;
        c->ew2[q] = nullptr;
    }
    c->hkeys = c->hvals = c->ew = nullptr;
    c->elo = c->ehi = nullptr;
    c->hcap = 0;
    LEM_CHECK(c, hipMalloc(&c->hkeys, cap * 8));
    LEM_CHECK(c, hipMalloc(&c->hvals, cap * 8));
    LEM_CHECK(c, hipMalloc(&c->elo, cap * 4));
    LEM_CHECK(c, hipMalloc(&c->ehi, cap * 4));
    LEM_CHECK(c, hipMalloc(&c->ew, cap * 8));
    for (int q = 0; q < 2; q++) {
        LEM_CHECK(c, hipMalloc(&c->elo2[q], cap * 4));
        LEM_CHECK(c, hipMalloc(&c->ehi2[q], cap * 4));
        LEM_CHECK(c, hipMalloc(&c->ew2[q], cap * 8));
    }
    c->hcap = cap;
    c->ecap = cap;
    return LEMHIP_OK;
}

static int ensure_labels(lemhip_ctx *c, long nl)
{
    if (nl <= c->lcap) return LEMHIP_OK;
    if (c->rmm) { (void)hipFree(c->rmm); (void)hipFree(c->seen); (void)hipFree(c->comp); (void)hipFree(c->cmax); }
    c->rmm = nullptr;
    c->seen = nullptr;
    c->comp = nullptr;
    c->cmax = nullptr;
    long cap = nl + nl / 4 + 1024;
    LEM_CHECK(c, hipMalloc(&c->rmm, cap * 8));
    LEM_CHECK(c, hipMalloc(&c->seen, cap));
    LEM_CHECK(c, hipMalloc(&c->comp, cap * 4));
    LEM_CHECK(c, hipMalloc(&c->cmax, cap * 8));
    c->lcap = cap;
    return LEMHIP_OK;
}

static int cutoff_components(lemhip_ctx *c, int nlab, int ne)
{
    long n = (long)nlab + 1;
    // second relaxation array: reuse the hash value table (>= 8*(nlab+1) slots)
    unsigned long long *r2 = c->hvals;
    k_fb_comp_init<<<grid1d(n), 256, 0, c->s>>>(n, c->comp, c->cmax);
    LEM_LAUNCHED(c);
    for (int it = 0;; ++it) {
        LEM_TRY(clear_flag(c));
        k_fb_comp_relax<<<grid1d(ne, 256, 1 << 30), 256, 0, c->s>>>(ne, c->elo, c->ehi, c->rmm, c->comp, &c->scal->flag);
        LEM_LAUNCHED(c);
        int f = 0;
        LEM_TRY(read_flag(c, &f));
        if (!f) break;
        if (it > nlab + 2) { c->err = "component labelling did not converge"; return LEMHIP_E_NOT_CONVERGED; }
    }
    k_fb_seed<<<grid1d(n), 256, 0, c->s>>>(n, c->rmm, c->comp, c->seen, r2);
    LEM_LAUNCHED(c);
    for (int it = 0;; ++it) {
        LEM_TRY(clear_flag(c));
        k_minimax_relax<<<grid1d(ne, 256, 1 << 30), 256, 0, c->s>>>(ne, c->elo, c->ehi, c->ew, r2, &c->scal->flag);
        LEM_LAUNCHED(c);
        int f = 0;
        LEM_TRY(read_flag(c, &f));
        if (!f) break;
        if (it > nlab + 2) { c->err = "cut-off spill heights did not converge"; return LEMHIP_E_NOT_CONVERGED; }
    }
    k_fb_max<<<grid1d(n), 256, 0, c->s>>>(n, c->rmm, c->comp, c->seen, r2, c->cmax);
    k_fb_apply<<<grid1d(n), 256, 0, c->s>>>(n, c->rmm, c->comp, c->seen, c->cmax);
    LEM_LAUNCHED(c);
    return LEMHIP_OK;
}

#define BV_KEEP_SHORT (1 << 20)
// Spill heights of the labels into c->rmm (initialised: label 0 -inf, the
// rest +inf) by Borůvka phases over the label-sorted edge list, whose length
// is in scal->nedges (at most `bound`, read with the first counts).  Two phases
// run between host reads, three where an empty one costs no more than a read
// (20 us on short label lists, 75 on the 8191x7003 DEM's): the kernels take the edge counts from the device and
// their grids from the last count the host knows.  A read leaves the device
// idle for about 15 us, as long as the phase itself on short lists (a step at
// 512^2 with seven reads fewer, these among them: 1.80 instead of 1.88 ms).
// jumps: pointer-jumping launches before each phase's walks; *over: a walk gave
// up, and the heights are of no use.
static int bv_phases(lemhip_ctx *c, long n, int bound, int jumps, bool *over)
{
    // per-label scratch: running maxima, chosen weights (parity 1) and label
    // 0's scalars in the hash value table, chosen edges and roots in the hash
    // key table (both >= 8 * (nlab + 1) entries of 8 bytes), chosen weights
    // (parity 0) in cmax
    unsigned long long *mv = c->hvals, *bw[2] = {c->cmax, c->hvals + n}, *st = c->hvals + 2 * n;
    uint32_t *be[2] = {reinterpret_cast<uint32_t *>(c->hkeys), reinterpret_cast<uint32_t *>(c->hkeys) + n};
    uint32_t *nxt = reinterpret_cast<uint32_t *>(c->hkeys) + 2 * n;
    k_bv_init<<<grid1d(n, 256, 2048), 256, 0, c->s>>>(n, c->comp, mv, bw[0], bw[1], be[0], be[1], st, c->seen,
                                                      c->labdem, jumps ? 0 : c->nslot, c->dsc,
                                                      jumps ? c->rmm : nullptr);
    LEM_LAUNCHED(c);
    const uint32_t *lo = c->elo, *hi = c->ehi;
    const unsigned long long *w = c->ew;
    const int *cnt = &c->scal->nedges;
    const int per = n <= (1 << 18) ? 3 : 2;
    // the profile slot times the kernels only, not the host reads between them
    for (int ph = 0, na = bound; na > 0;) {
        for (int q = 0; q < per; q++, ph++) {
            const int p = ph & 1;
            const int ge = grid1d(na, 256, 1 << 30);
            uint32_t *lo2 = c->elo2[p], *hi2 = c->ehi2[p];
            unsigned long long *w2 = c->ew2[p];
            int *kept = &c->scal->kept[p];
            prof_begin(c, PROF_MM_K);
            k_bv_min_w<<<ge, 256, 0, c->s>>>(cnt, lo, hi, w, c->comp, bw[p]);
            k_bv_min_e<<<ge, 256, 0, c->s>>>(cnt, lo, hi, w, c->comp, bw[p], be[p]);
            k_bv_hook<<<grid1d(n), 256, 0, c->s>>>(n, lo, hi, c->comp, be[p], nxt, kept);
            for (int j = 0; j < jumps; j++) k_bv_jump<<<grid1d(n), 256, 0, c->s>>>(n, nxt);
            k_bv_labels<<<grid1d(n), 256, 0, c->s>>>(n, c->comp, bw[p], be[p], nxt, mv, c->rmm, st + 2 * p,
                                                      st + 2 * (p ^ 1), bw[p ^ 1], be[p ^ 1], &c->scal->flag);
            if (na <= BV_KEEP_SHORT)
                k_bv_keep<4><<<grid_chunks(na, 8192, 4), 256, 0, c->s>>>(cnt, lo, hi, w, c->comp, lo2, hi2, w2, kept);
            else
                k_bv_keep<COMPACT_ITEMS><<<grid_chunks(na), 256, 0, c->s>>>(cnt, lo, hi, w, c->comp, lo2, hi2, w2,
                                                                            kept);
            prof_end(c, PROF_MM_K, 5 + jumps);
            LEM_LAUNCHED(c);
            lo = lo2; hi = hi2; w = w2;
            cnt = kept;
        }
        LEM_TRY(read_scalars(c));
        c->h_nedges = c->hscal->nedges;
        *over = c->hscal->flag != 0;
        if (*over) return LEMHIP_OK;
        const int nk = c->hscal->kept[(ph - 1) & 1];
        // every component with an outgoing edge joins another each phase, so
        // the components with edges at least halve
        if (nk >= na && ph > per) { c->err = "spill-height phases made no progress"; return LEMHIP_E_NOT_CONVERGED; }
        na = nk;
        if (ph > 64) { c->err = "spill-height phases did not converge"; return LEMHIP_E_NOT_CONVERGED; }
    }
    return LEMHIP_OK;
}

// The phases with walks alone, and if a path was too long for them, once more
// with as many jumps as the longest path can need.
static int spill_heights(lemhip_ctx *c, int nlab, int bound)
{
    const long n = (long)nlab + 1;
    c->h_nedges = 0;
    if (bound <= 0) return LEMHIP_OK;
    bool over = false;
    LEM_TRY(bv_phases(c, n, bound, 0, &over));
    if (!over) return LEMHIP_OK;
    int jumps = 1;
    while ((1L << jumps) < n) jumps++;
    LEM_TRY(clear_flag(c));
    LEM_TRY(bv_phases(c, n, bound, jumps, &over));
    if (over) { c->err = "spill-height component pointers form a cycle"; return LEMHIP_E_NOT_CONVERGED; }
    return LEMHIP_OK;
}

static int raise_surface(lemhip_ctx *c)
{
    k_raise<<<grid1d(c->N), 256, 0, c->s>>>(c->N, c->mask, c->ws, c->rmm, c->dem, c->demid, c->dsc, c->z2);
    LEM_LAUNCHED(c);
    return LEMHIP_OK;
}


// floodingDriver (routeflow.cu:202-676) up to the raised surface in c->z2.
// *sinks: whether pass 1 left any, read with the label count; if not, nothing is
// flooded.
static int flooding(lemhip_ctx *c, int ncand1, int *sinks)
{
    long N = c->N;
    int W = c->W, H = c->H;
    // labels
    k_sink_flags<<<grid2d(W, H), 256, 0, c->s>>>(W, H, c->mask, c->SFD, c->demid, c->ddesc, c->scan_tmp);
    LEM_LAUNCHED(c);
    size_t need = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, need, c->scan_tmp, c->ws, (int)N, c->s);
    if (need > c->cub_bytes) {
        if (c->cub_tmp) (void)hipFree(c->cub_tmp);
        c->cub_tmp = nullptr;
        LEM_CHECK(c, hipMalloc(&c->cub_tmp, need));
        c->cub_bytes = need;
    }
    // prefix lands in ws, then k_init_ws rewrites ws in place from it: use z2 as the prefix buffer instead
    int *prefix = reinterpret_cast<int *>(c->z2);
    LEM_CHECK(c, hipcub::DeviceScan::ExclusiveSum(c->cub_tmp, need, c->scan_tmp, prefix, (int)N, c->s));
    k_init_ws<<<grid2d(W, H), 256, 0, c->s>>>(W, H, c->mask, c->SFD, prefix, c->demid, c->ddesc, c->ws, c->labdem,
                                              &c->scal->nlabels);
    // sink merge over the sinks that have an equal-height neighbour (list in the
    // prefix buffer, free after k_init_ws); the first rounds run before the
    // host knows of any
    int *mlist = reinterpret_cast<int *>(c->z2);
    k_merge_list<<<grid1d(ncand1, 256, 4096), 256, 0, c->s>>>(c->cand, ncand1, c->SFD, c->dmask, mlist,
                                                             &c->scal->ncand);
    LEM_LAUNCHED(c);
    for (long it = 0;; it += 4) {
        const int gm = it ? grid1d(c->hscal->ncand, 256, 1 << 30) : grid1d(ncand1, 256, 256);
        if (it) LEM_TRY(clear_flag(c));
        for (int q = 0; q < 4; q++)
            k_sink_merge<<<gm, 256, 0, c->s>>>(W, H, mlist, &c->scal->ncand, c->SFD, c->dem, c->ws, &c->scal->flag);
        LEM_LAUNCHED(c);
        LEM_TRY(read_scalars(c));
        *sinks = c->hscal->sinks_pass1;
        if (*sinks == 0) return LEMHIP_OK;
        if (!c->hscal->flag) break;
        if (it / 4 > (long)c->hscal->ncand + 2) { c->err = "sink merge did not converge"; return LEMHIP_E_NOT_CONVERGED; }
    }
    const int nlab = c->hscal->nlabels;
    c->h_nlab = nlab;
    // watershed labels: one jump over every cell, two or three where basins are
    // large and so paths long, then each walks the rest.  On the smooth 2000x1500
    // DEM (few basins) one jump leaves depression routing at 0.72 ms, two at 0.41,
    // three at 0.37 (1.35 with one link and no progress left); on a straight
    // valley of 4096 rows (2900 cells a basin) one leaves it at 1.49 ms, two at
    // 1.05; on 8191x7003 (250 cells a basin) a second costs 0.08 of 4.11 ms.
    // A walk takes at most 256 links, after three jumps 128.  Where that is not
    // enough, WS_JUMPS jumps of one link each, which double what a pointer
    // spans, and more walks follow until every cell has its label: a valley
    // winding over 4096^2 2.9 ms, 4.6 with many small basins beside it (89 and
    // 1740 with walks to the end; 2.0 at 64 links, but then 0.1 more on the
    // straight valley)
#define WS_JUMPS 8
    const long basin = N / (nlab + 1L);   // cells of one, on average
    const int limit = basin > 4096 ? 128 : 256;
    for (int q = basin > 4096 ? 3 : basin > 1024 ? 2 : 1; q > 0; q--)
        k_jump<4><<<grid1d(N), 256, 0, c->s>>>(N, c->mask, c->ws, &c->scal->flag, &c->scal->nedges);
    k_jump_walk<<<grid1d(N), 256, 0, c->s>>>(N, c->mask, c->ws, limit, &c->scal->flag);
    LEM_LAUNCHED(c);
    // edges: block-distinct pairs appended, sorted by pair, reduced to the
    // minimum weight per pair; the list comes out sorted by label (the
    // Borůvka phases read neighbouring labels' components from the same
    // lines, and their ties are broken by position in this order)
    LEM_TRY(ensure_labels(c, (long)nlab + 1));
    int B = 1;
    while ((1L << B) <= (long)nlab) B++;
    long want = 8L * (nlab + 1);
    if (want < 1024) want = 1024;
    long np = 0;
    for (int attempt = 0, walks = 0;; ++attempt) {
        LEM_TRY(ensure_hash(c, want));
        if (attempt) LEM_CHECK(c, hipMemsetAsync(&c->scal->nedges, 0, sizeof(int), c->s));
        dim3 blk(64, 4), grd((W + 63) / 64, (H + 4 * EDGE_RG - 1) / (4 * EDGE_RG));
        k_edges_emit<<<grd, blk, 0, c->s>>>(W, H, c->mask, c->ws, c->dem, c->demid, c->hkeys, c->hvals, c->hcap,
                                            &c->scal->nedges, B, &c->scal->flag);
        LEM_LAUNCHED(c);
        LEM_TRY(read_scalars(c));
        if (c->hscal->flag) {   // paths longer than one launch's walks
            for (int more = 1; more;) {
                if (++walks > 8) { c->err = "watershed pointer jumping did not converge"; return LEMHIP_E_NOT_CONVERGED; }
                for (int q = 0; q < WS_JUMPS; q++)
                    k_jump<1><<<grid1d(N), 256, 0, c->s>>>(N, c->mask, c->ws, &c->scal->flag, &c->scal->nedges);
                k_jump_walk<<<grid1d(N), 256, 0, c->s>>>(N, c->mask, c->ws, limit, &c->scal->flag);
                LEM_LAUNCHED(c);
                LEM_TRY(read_flag(c, &more));
            }
            continue;
        }
        np = c->hscal->nedges;
        if (np <= c->hcap) break;
        want = np + np / 4;
        if (attempt > 8) { c->err = "edge list overflow"; return LEMHIP_E_NOMEM; }
    }
    // labels cut off from label 0 (NaN heights only) raise the flag `cut`, read
    // with the next pass's first counts: the surface is raised before it is known
    int *cut = &reinterpret_cast<PlatCtl *>(c->pl_ctl)->cut;
    k_minimax_init<<<grid1d(std::max(nlab + 1, c->nslot)), 256, 0, c->s>>>(nlab + 1, c->rmm, c->seen, c->nslot, c->dsc,
                                                                          &c->scal->flag, cut);
    LEM_LAUNCHED(c);
    if (np > 0) {
        unsigned long long *skeys = c->ew2[0], *svals = c->ew2[1];
        size_t need3 = 0, need4 = 0;
        (void)hipcub::DeviceRadixSort::SortPairs(nullptr, need3, c->hkeys, skeys, c->hvals, svals, (int)np, 0, 2 * B,
                                                 c->s);
        (void)hipcub::DeviceReduce::ReduceByKey(nullptr, need4, skeys, c->hkeys, svals, c->hvals, &c->scal->nedges,
                                                hipcub::Min(), (int)np, c->s);
        if (need4 > need3) need3 = need4;
        if (need3 > c->cub_bytes) {
            if (c->cub_tmp) (void)hipFree(c->cub_tmp);
            c->cub_tmp = nullptr;
            LEM_CHECK(c, hipMalloc(&c->cub_tmp, need3));
            c->cub_bytes = need3;
        }
        size_t t3 = c->cub_bytes;
        LEM_CHECK(c, hipcub::DeviceRadixSort::SortPairs(c->cub_tmp, t3, c->hkeys, skeys, c->hvals, svals, (int)np, 0,
                                                         2 * B, c->s));
        t3 = c->cub_bytes;
        LEM_CHECK(c, hipcub::DeviceReduce::ReduceByKey(c->cub_tmp, t3, skeys, c->hkeys, svals, c->hvals,
                                                        &c->scal->nedges, hipcub::Min(), (int)np, c->s));
        k_edges_decode<<<((int)np + 255) / 256, 256, 0, c->s>>>(&c->scal->nedges, c->hkeys, c->hvals, B, c->elo, c->ehi,
                                                                c->ew, c->seen, c->labdem, c->dsc);
        LEM_LAUNCHED(c);
    }

    LEM_TRY(spill_heights(c, nlab, (int)np));
    const int ne = c->h_nedges;
    if (ne > 0) k_fb_unreached<<<grid1d(ne, 256, 1 << 30), 256, 0, c->s>>>(ne, c->elo, c->ehi, c->rmm, cut);
    return raise_surface(c);
}

// Times the plateau pass with every rounds-per-launch candidate on the same
// surface (the pass is idempotent: it rebuilds directions, distances and marks
// from the surface) and keeps the fastest.
template <typename TS>
static int tune_plateau(lemhip_ctx *c, const double *zs, TS *slopes)
{
    static const int KS[3] = {4, 8, 16};
    // each choice timed twice, in the order 8 4 16 16 4 8, keeping its
    // faster time: a context tuned beside others sees their phases change
    // between its timings, and one timing per choice picked 4 on some boxes
    static const int ORDER[6] = {1, 0, 2, 2, 0, 1};
    hipEvent_t e0, e1;
    LEM_CHECK(c, hipEventCreate(&e0));
    LEM_CHECK(c, hipEventCreate(&e1));
    for (int q = 0; q < 3; q++) c->tune_ms[8 + q] = 1e30;
    for (int o = 0; o < 6; o++) {
        const int q = ORDER[o];
        c->plat_k = KS[q];
        int n = 0, r = 0;
        LEM_CHECK(c, hipEventRecord(e0, c->s));
        LEM_TRY(directions_and_plateaus<TS>(c, zs, slopes, &n, &r));
        LEM_CHECK(c, hipEventRecord(e1, c->s));
        LEM_CHECK(c, hipEventSynchronize(e1));
        float ms = 0.f;
        LEM_CHECK(c, hipEventElapsedTime(&ms, e0, e1));
        if (ms < c->tune_ms[8 + q]) c->tune_ms[8 + q] = ms;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    float best = 1e30f;
    int bestk = 8;
    for (int q = 0; q < 3; q++)
        if ((float)c->tune_ms[8 + q] < best) { best = (float)c->tune_ms[8 + q]; bestk = KS[q]; }
    // 8 rounds per launch fit the tile's region best (one region row per
    // wave, five cells per thread): another count only when clearly faster,
    // since contexts tuned side by side time each other's traffic too
    if (bestk != 8 && best > 0.9f * (float)c->tune_ms[9]) bestk = 8;
    c->plat_k = bestk;
    c->tune_plat_pending = false;
    return LEMHIP_OK;
}

template <typename TS>
static int fd_phase_t(lemhip_ctx *c, int iter)
{
    (void)iter;
    long N = c->N;
    // lowest cell for the outlet check, taken on the unadjusted surface
    prof_begin(c, PROF_FD);
    LEM_TRY(lem_slot_lowest(c, c->dem, 0, c->nslot));
    // pass 1 on the unraised surface; slopes keep these values
    int n1 = 0, r1 = 0;
    LEM_TRY(directions_and_plateaus<TS>(c, c->dem, reinterpret_cast<TS *>(c->slopes), &n1, &r1));
    k_slots_sinks_init<<<(c->nslot + 255) / 256, 256, 0, c->s>>>(c->nslot, c->dsc, c->scal);
    if (n1 > 0) {
        k_count_sinks<<<grid1d(n1, 256, 2048), 256, 0, c->s>>>(c->cand, n1, c->SFD, c->demid, c->nslot, c->dsc,
                                                                &c->scal->sinks_pass1);
        LEM_LAUNCHED(c);
    }
    c->h_rounds1 = r1;
    c->h_rounds2 = 0;
    c->h_nlab = 0;
    c->h_nedges = 0;
    prof_begin(c, PROF_FLOOD);
    int sinks = 0;
    if (n1 > 0) LEM_TRY(flooding(c, n1, &sinks));
    if (sinks > 0)
        k_slots_sinkcount_fin<<<(c->nslot + 255) / 256, 256, 0, c->s>>>(c->ddesc, c->nslot, c->dsc);
    prof_end(c, PROF_FLOOD);
    if (sinks == 0) {
        c->h_nlab = 0;
        k_slots_sinkcount_init<<<(c->nslot + 255) / 256, 256, 0, c->s>>>(c->nslot, c->dsc);
    } else {
        int n2 = 0, r2 = 0;
        bool cut = false;
        LEM_TRY(directions_and_plateaus<TS>(c, c->z2, (TS *)nullptr, &n2, &r2, &cut));
        if (cut) {
            prof_begin(c, PROF_FLOOD);
            LEM_TRY(cutoff_components(c, c->h_nlab, c->h_nedges));
            LEM_TRY(raise_surface(c));
            prof_end(c, PROF_FLOOD, 0);
        }
        if (c->tune_plat_pending) LEM_TRY(tune_plateau<TS>(c, c->z2, (TS *)nullptr));
        if (cut) LEM_TRY(directions_and_plateaus<TS>(c, c->z2, (TS *)nullptr, &n2, &r2));
        c->h_rounds2 = r2;
    }
    k_merge<<<grid1d(N), 256, 0, c->s>>>(N, c->p.flowdirectiontype, c->mask, c->fd, c->SFD);
    k_slots_outlet_adjust<<<(c->nslot + 255) / 256, 256, 0, c->s>>>(c->dem, c->fd, c->ddesc, c->nslot, c->dsc);
    LEM_LAUNCHED(c);
    prof_end(c, PROF_FD);
    return LEMHIP_OK;
}

int lem_fd_phase(lemhip_ctx *c, int iter)
{
    if (c->prec == LEMHIP_FP64) return fd_phase_t<double>(c, iter);
    return fd_phase_t<float>(c, iter);
}
