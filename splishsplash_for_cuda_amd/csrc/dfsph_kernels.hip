// dfsph_kernels.hip -- hand-written gfx950 kernels of the DFSPH time step.
//
// One thread per particle, particles in cell-sorted order, kBlock-thread
// blocks (512) with the XCD-aware block remap of dfsph_device.hpp.  Every kernel
// cites the reference kernel(s) it replaces (paths relative to the
// reference repository root).
#include <hip/hip_ext.h>

#include "dfsph_device.hpp"
#include "dfsph_launch.hpp"

namespace dfsph {

// ------------------------------------------------------------------------
// small utilities
// ------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_fill_f32(float* p, float v, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Loop-control init (the host-side locals of cuda_divergenceSolve /
// cuda_pressureSolve, DFSPH_core_cuda.cu:785-828, 1338-1378).
// eta = max_error * 0.01 * rho0 (/ h for the divergence solver).
__global__ void k_nbr_ctl_init(DevCtl* c)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->max_seen = 0;
        c->overflow = 0;
        c->nbr_fluid = 0;
        c->nbr_boundary = 0;
        c->nbr_fluid_unstaged = 0;
        c->unstaged_blocks = 0;
    }
}

static __device__ void time_fill(DevTime* t, double h, double hf, double hp)
{
    t->hd = h; t->hfd = hf; t->hpd = hp;
    t->h = (float)h; t->h_future = (float)hf; t->h_past = (float)hp;
    t->inv_h = (float)(1.0 / h);
    t->inv_h_future = (float)(1.0 / hf);
}

// Thread-level: copy the loop and step state into the host record, then
// release its sequence number at system scope.
__device__ void publish(const Publish& pub, const SolveCtl* sc)
{
    HostRecord* r = pub.rec;
    r->sc = *sc;
    r->tm = *pub.t;
    r->max_seen = pub.dc->max_seen;
    r->overflow = pub.dc->overflow;
    r->unstaged_blocks = pub.dc->unstaged_blocks;
    r->escaped = pub.dc->escaped;
    r->nbr_fluid = pub.dc->nbr_fluid;
    r->nbr_boundary = pub.dc->nbr_boundary;
    r->nbr_fluid_unstaged = pub.dc->nbr_fluid_unstaged;
    __threadfence_system();
    __hip_atomic_store(&r->seq, pub.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A count the host waits for, published as the loop state is.
__global__ void k_publish_count(const uint32_t* count, HostRecord* r, uint32_t seq)
{
    if (threadIdx.x == 0) {
        r->count = *count;
        __threadfence_system();
        __hip_atomic_store(&r->count_seq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// DFSPHCData::reset time bookkeeping (DFSPH_c_arrays_structure.cpp:1000-1004)
__global__ void k_time_reset(DevTime* t, double h)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        time_fill(t, h, h, h);
        t->ratio = 1.0f; t->ratio2 = 1.0f;
        t->time = 0.0;
    }
}

// DFSPHCData::updateTimeStep (DFSPH_c_arrays_structure.cpp:1100-1106).  mode 0: the
// given h_future; mode 1: the CFL estimate of cuda_CFL (DFSPH_core_cuda.cu:3380-3387),
// h = cfl_factor * 0.4 * 2r / sqrt(max |v + a h|^2) clamped to [dt_min, dt_max],
// the maximum taken here from the XSPH sweep's nparts block maxima; mode 2: keep
// the current h (constant step, DFSPH_CUDA.cpp:302-306).
__global__ __launch_bounds__(kBlock) void k_time_update(DevTime* t, double hf, DevCtl* ctl, const float* partial,
                                                        uint32_t nparts, int mode, double cfl_factor, double diameter,
                                                        double dt_min, double dt_max, double cfl_seed)
{
    __shared__ float lds4[kBlock / 64];
    if (mode == 1) {
        constexpr uint32_t kBatch = 8;
        float mm = 0.0f;
        for (uint32_t k0 = threadIdx.x; k0 < nparts; k0 += kBatch * kBlock) {
            float v[kBatch];
#pragma unroll
            for (uint32_t u = 0; u < kBatch; ++u) {
                const uint32_t k = k0 + u * kBlock;
                v[u] = k < nparts ? partial[k] : 0.0f;
            }
#pragma unroll
            for (uint32_t u = 0; u < kBatch; ++u) mm = fmaxf(mm, v[u]);
        }
        mm = wave_max(mm);
        if ((threadIdx.x & 63) == 0) lds4[threadIdx.x >> 6] = mm;
        __syncthreads();
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (mode == 2) hf = t->hd;
        if (mode == 1) {
            float bm = lds4[0];
            for (int k = 1; k < kBlock / 64; ++k) bm = fmaxf(bm, lds4[k]);
            ctl->cfl_max = bm;
            double m = (double)bm;
            m = m > cfl_seed ? m : cfl_seed;
            double h = cfl_factor * 0.4 * (diameter / sqrt(m));
            if (!(h < dt_max)) h = dt_max;
            if (h < dt_min) h = dt_min;
            hf = h;
        }
        const double h = t->hd;
        time_fill(t, h, hf, t->hpd);
        t->ratio = (float)(h / hf);
        t->ratio2 = (float)((h * h) / (hf * hf));
    }
}

// resume from a snapshot: h, h_past, time; h_future = h and the ratios of the
// last updateTimeStep (h_past / h)
__global__ void k_time_set(DevTime* t, double h, double hp, double time)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        time_fill(t, h, h, hp);
        t->ratio = (float)(hp / h);
        t->ratio2 = (float)((hp * hp) / (h * h));
        t->time = time;
    }
}

// DFSPHCData::onSimulationStepEnd (DFSPH_c_arrays_structure.cpp:1108-1118) and the
// TimeManager advance time += h (DFSPH_CUDA.cpp:449-452, with the new h).
__global__ void k_time_step_end(DevTime* t, Publish pub)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const double hp = t->hd, h = t->hfd;
        time_fill(t, h, h, hp);
        t->time += h;
        if (pub.rec) publish(pub, &pub.dc->dens);
    }
}

// ------------------------------------------------------------------------
// exclusive scan of uint32 (replaces cub::DeviceScan::ExclusiveSum,
// DFSPH_core_cuda.cu:1920): tiles of 2048 in LDS, deterministic.
// ------------------------------------------------------------------------
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;

__global__ __launch_bounds__(kBlock) void k_scan_tiles(uint32_t* in, uint32_t* out, uint32_t n,
                                                        uint32_t* tile_sums, int clear_in)
{
    __shared__ uint32_t tile[kScanTile];
    __shared__ uint32_t wsum[kBlock / 64];
    const uint32_t base = blockIdx.x * kScanTile;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t g = base + k * kBlock + threadIdx.x;
        tile[k * kBlock + threadIdx.x] = g < n ? in[g] : 0u;
        if (clear_in && g < n) in[g] = 0u;     // a histogram left zeroed for its next use
    }
    __syncthreads();
    uint32_t loc[kScanItems];
    uint32_t run = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        loc[k] = run;
        run += tile[threadIdx.x * kScanItems + k];
    }
    const uint32_t incl = wave_incl_scan_u(run);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63) wsum[w] = incl;
    __syncthreads();
    uint32_t woff = 0;
    for (int k = 0; k < w; ++k) woff += wsum[k];
    const uint32_t excl = woff + incl - run;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) tile[threadIdx.x * kScanItems + k] = excl + loc[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t g = base + k * kBlock + threadIdx.x;
        if (g < n) out[g] = tile[k * kBlock + threadIdx.x];
    }
    if (threadIdx.x == kBlock - 1) {
        uint32_t tot = 0;
        for (int k = 0; k < kBlock / 64; ++k) tot += wsum[k];
        tile_sums[blockIdx.x] = tot;
    }
}

// The tile's offset is the sum of the preceding tile sums, which each block
// adds up itself (grids of up to kScanDirect tiles): no scan of the sums.
constexpr uint32_t kScanDirect = 4096;
__global__ __launch_bounds__(kBlock) void k_scan_add_direct(uint32_t* out, uint32_t n, const uint32_t* tile_sums)
{
    __shared__ uint32_t ws[kBlock / 64];
    uint32_t acc = 0;
    for (uint32_t t = threadIdx.x; t < blockIdx.x; t += kBlock) acc += tile_sums[t];
    acc = wave_sum_u(acc);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = acc;
    __syncthreads();
    uint32_t off = 0;
#pragma unroll
    for (int k = 0; k < kBlock / 64; ++k) off += ws[k];
    const uint32_t base = blockIdx.x * kScanTile;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t g = base + k * kBlock + threadIdx.x;
        if (g < n) out[g] += off;
    }
}

__global__ __launch_bounds__(kBlock) void k_scan_add(uint32_t* out, uint32_t n, const uint32_t* tile_off)
{
    const uint32_t off = tile_off[blockIdx.x];
    const uint32_t base = blockIdx.x * kScanTile;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t g = base + k * kBlock + threadIdx.x;
        if (g < n) out[g] += off;
    }
}

// ------------------------------------------------------------------------
// neighbor search (cuda_neighborsSearch, DFSPH_core_cuda.cu:1833-2129, 2219-2531)
// ------------------------------------------------------------------------

// DFSPH_computeGridIdx_kernel (DFSPH_core_cuda.cu:1833-1848): cell id and the
// particle's arrival slot in its cell.  Particles outside the grid are
// clamped into the border cells.
// Consecutive particles mostly share a cell (the previous step left them in
// cell order), so each run of equal keys in a wave takes its slots with one
// atomic: the run's first lane adds the run length and the others offset from
// the returned base.
__global__ __launch_bounds__(kBlock) void k_cell_hist(SimConst c, const float4* pos, uint32_t n, uint32_t* key,
                                                      uint32_t* slot, uint32_t* hist)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool act = i < n;
    uint32_t k = kKeyInvalid;
    if (act) {
        const float4 p = pos[i];
        k = cell_id(c, p.x, p.y, p.z);
    }
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t prev = __shfl_up(k, 1, 64);
    const bool head = lane == 0u || prev != k;
    const uint64_t heads = __ballot(head);
    const uint64_t upto = lane == 63u ? ~0ull : ((2ull << lane) - 1ull);   // lanes 0..lane
    const uint32_t h = 63u - (uint32_t)__clzll((long long)(heads & upto));  // my run's first lane
    const uint64_t after = heads & ~upto;
    const uint32_t next = after ? (uint32_t)__ffsll((long long)after) - 1u : 64u;
    uint32_t base = 0;
    if (act && head) base = atomicAdd(hist + k, next - lane);
    base = __shfl(base, (int)h, 64);
    if (act) {
        key[i] = k;
        slot[i] = base + (lane - h);
    }
}

// DFSPH_CountingSortIds_kernel (DFSPH_core_cuda.cu:1851-1858)
__global__ void k_scatter_perm(const uint32_t* key, const uint32_t* slot, const uint32_t* cstart,
                               uint32_t n, uint32_t* perm)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    perm[cstart[key[i]] + slot[i]] = i;
}

// The arrival slots come from atomics, so the order inside a cell varies from
// run to run (DFSPH_core_cuda.cu:1845-1846).  A particle's place is its cell's
// start plus the number of the cell's entries with a smaller original index,
// which makes the counting sort stable and the whole step bit-reproducible.
// The consumers of the order count it themselves, one thread per entry: the
// cell's entries are in a cache line or two that the neighbors read too,
// and no pass sorts them in memory (an insertion sort with a thread per cell
// took 28 us of a 4.19 M particle search, 80 us with 200k particles where
// spray crowds some cells).
struct CellOrder {
    const uint32_t* __restrict__ key;
    const uint32_t* __restrict__ cstart;
    const uint32_t* __restrict__ perm;   // perm: the entries of each cell in arrival order
};

__device__ __forceinline__ uint32_t ordered_place(const CellOrder& o, uint32_t i)
{
    const uint32_t c = o.key[i], s = o.cstart[c], e = o.cstart[c + 1];
    uint32_t rank = 0, q = s;
    for (; q + 4u <= e; q += 4u) {
        const uint32_t a0 = o.perm[q], a1 = o.perm[q + 1u], a2 = o.perm[q + 2u], a3 = o.perm[q + 3u];
        rank += (a0 < i ? 1u : 0u) + (a1 < i ? 1u : 0u) + (a2 < i ? 1u : 0u) + (a3 < i ? 1u : 0u);
    }
    for (; q < e; ++q) rank += o.perm[q] < i ? 1u : 0u;
    return s + rank;
}

// the stable order itself, for searches and scans that read through it
__global__ void k_order_perm(uint32_t n, CellOrder o, uint32_t* out)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t i = o.perm[k];
    out[ordered_place(o, i)] = i;
}

// cuda_sortData (DFSPH_core_cuda.cu:2057-2129): one gather of every persistent
// per-particle field into the alternate buffers (no device-to-device copies).
__device__ __forceinline__ void copy_fluid(const FluidPtrs& a, uint32_t from, const FluidPtrs& b, uint32_t to)
{
    b.pos[to] = a.pos[from];
    b.vel[to] = a.vel[from];
    b.kap[to] = a.kap[from];
    b.kapv[to] = a.kapv[from];
    b.ktot[to] = a.ktot[from];
    b.kvtot[to] = a.kvtot[from];
    b.id[to] = a.id[from];
    b.tag[to] = a.tag[from];
}

__global__ void k_gather_fluid(uint32_t n, CellOrder o, FluidPtrs in, FluidPtrs out)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t i = o.perm[k];
    // the record is in flight while its place is counted
    const float4 p = in.pos[i], v = in.vel[i];
    const float ka = in.kap[i], kv = in.kapv[i], kt = in.ktot[i], kvt = in.kvtot[i];
    const uint32_t id = in.id[i], tag = in.tag[i];
    const uint32_t to = ordered_place(o, i);
    out.pos[to] = p;
    out.vel[to] = v;
    out.kap[to] = ka;
    out.kapv[to] = kv;
    out.ktot[to] = kt;
    out.kvtot[to] = kvt;
    out.id[to] = id;
    out.tag[to] = tag;
}

// the boundary set's records (positions, and velocities when given) in cell order
__global__ void k_gather_boundary(uint32_t n, CellOrder o, const float4* in, float4* out, const float4* vin,
                                  float4* vout)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t i = o.perm[k], to = ordered_place(o, i);
    out[to] = in[i];
    if (vin) vout[to] = vin[i];
}

// Appends list entries to a particle's blocked-interleaved list: entries
// shift into a 16-byte register group from the top (a funnel shift per word)
// and each full group is one store at the running group pointer.
struct ListWriter16 {
    uint4* out;                    // the particle's next group
    uint32_t cap;                  // groups are cap apart
    uint32_t n = 0;                // entries pushed
    uint32_t w0 = 0, w1 = 0, w2 = 0, w3 = 0;
    __device__ __forceinline__ void shift_in(uint32_t v)
    {
        w0 = __builtin_amdgcn_alignbit(w1, w0, 16);
        w1 = __builtin_amdgcn_alignbit(w2, w1, 16);
        w2 = __builtin_amdgcn_alignbit(w3, w2, 16);
        w3 = __builtin_amdgcn_alignbit(v, w3, 16);
    }
    __device__ __forceinline__ void push(uint32_t v)  // 16 bits
    {
        shift_in(v);
        ++n;
        if ((n & 7u) == 0u) { *out = make_uint4(w0, w1, w2, w3); out += cap; }
    }
    __device__ __forceinline__ void finish()
    {
        if (n & 7u) {
            for (uint32_t k = n & 7u; k < 8u; ++k) shift_in(0u);
            *out = make_uint4(w0, w1, w2, w3);
        }
    }
};

struct ListWriter32 {
    uint4* out;
    uint32_t cap;
    uint32_t n = 0;
    uint32_t w0 = 0, w1 = 0, w2 = 0, w3 = 0;
    __device__ __forceinline__ void shift_in(uint32_t v)
    {
        w0 = w1;
        w1 = w2;
        w2 = w3;
        w3 = v;
    }
    __device__ __forceinline__ void push(uint32_t v)
    {
        shift_in(v);
        ++n;
        if ((n & 3u) == 0u) { *out = make_uint4(w0, w1, w2, w3); out += cap; }
    }
    __device__ __forceinline__ void finish()
    {
        if (n & 3u) {
            for (uint32_t k = n & 3u; k < 4u; ++k) shift_in(0u);
            *out = make_uint4(w0, w1, w2, w3);
        }
    }
};

// Neighbor-search tables.  A block's set cells are the grid cells within one
// cell of its own cells, in (y, z, x) order.  They are collected as one 64-bit
// mask of x positions per row (y, z) of their bounding box; a cell's number is
// its row's first number plus the marked cells before it in the row, so the
// three cells x-1..x+1 of any row are consecutive: one contiguous range of
// the set per row.
// LDS of the search with 512-particle blocks: 2688 staged positions (12 B each)
// and 512 set cells take 40 KB (larger sets pass through the stage in windows).
// Sparse blocks (spray) have many cells and few particles: tables of up to
// kBigCells cells take the upper half of the stage, the lower one holds positions.
#ifndef DFSPH_NBR_STAGE
#define DFSPH_NBR_STAGE (DFSPH_BLOCK == 512 ? 2688 : 2048)
#endif
constexpr uint32_t kNbrStage = DFSPH_NBR_STAGE;   // set positions staged in LDS by the search
static_assert(kNbrStage % 16 == 0, "halves, and rows in whole words");
constexpr uint32_t kHalfStage = kNbrStage / 2;
// Rows (y, z) of a tabled set's bounding box.  34 x 34 of them hold the set of a
// block that runs from one octant of a 32-cell cube to the next (1008 did not:
// the few such blocks searched cell by cell, and of 258k particles the whole
// search waited for them, 82 us against 54).
constexpr uint32_t kSetRows = kHalfStage * 9 / 10 & ~1u;
#ifndef DFSPH_SET_CELLS
#define DFSPH_SET_CELLS (DFSPH_BLOCK == 512 ? 512 : 384)
#endif
constexpr uint32_t kSetCells = DFSPH_SET_CELLS;   // set cells with a full stage
constexpr uint32_t kBigCells = kHalfStage - 1;    // set cells with half a stage
// Box place of a set cell in a word, x | z << 6 | y << 16, and the widest box whose
// places it holds (kSetRows bounds z too, but only in boxes of two rows in y and more).
constexpr uint32_t kPlaceZ = 6, kPlaceY = 16;
constexpr uint32_t kBoxW = 1u << kPlaceZ, kBoxD = 1u << (kPlaceY - kPlaceZ);
static_assert(kBoxW == 64, "a row's mask has 64 bits");
static_assert(kSetRows <= 1u << (32 - kPlaceY), "y of a box place");
constexpr uint32_t kNoRow = 0xffffffffu;
constexpr int kIntMax = 0x7fffffff;

__device__ __forceinline__ int wave_min_i(int v)
{
    auto op = [](uint32_t a, uint32_t b) { return (uint32_t)min((int)a, (int)b); };
    return __builtin_amdgcn_readlane((int)wave_prefix_dpp((uint32_t)v, (uint32_t)kIntMax, op), 63);
}

__device__ __forceinline__ int wave_max_i(int v)
{
    auto op = [](uint32_t a, uint32_t b) { return (uint32_t)max((int)a, (int)b); };
    return __builtin_amdgcn_readlane((int)wave_prefix_dpp((uint32_t)v, (uint32_t)(-kIntMax - 1), op), 63);
}

__device__ __forceinline__ uint32_t wave_total_u(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_scan_u(v), 63);
}

// m = 2 m + (d < limit) for four distances in turn: the compares' carries join the
// shifts, two vector instructions per candidate (false for a NaN distance).
// A vector instruction has to wait two others before it reads a scalar
// register that one has written, so the compares come first, into registers of
// their own: three instructions lie between each and the sum that reads it.
// (Written as m + m + (d < limit) a candidate takes three: a search of 4.19 M
// particles 486 us, with this 475.)
__device__ __forceinline__ uint32_t shift_in_less(uint32_t m, float d0, float d1, float d2, float d3, float limit)
{
    unsigned long long c0, c1, c2;
    asm("v_cmp_gt_f32_e64 %1, %8, %4\n\t"
        "v_cmp_gt_f32_e64 %2, %8, %5\n\t"
        "v_cmp_gt_f32_e64 %3, %8, %6\n\t"
        "v_cmp_gt_f32_e32 vcc, %8, %7\n\t"
        "v_addc_co_u32_e64 %0, %1, %0, %0, %1\n\t"
        "v_addc_co_u32_e64 %0, %2, %0, %0, %2\n\t"
        "v_addc_co_u32_e64 %0, %3, %0, %0, %3\n\t"
        "v_addc_co_u32_e32 %0, vcc, %0, %0, vcc"
        : "+v"(m), "=&s"(c0), "=&s"(c1), "=&s"(c2)
        : "v"(d0), "v"(d1), "v"(d2), "v"(d3), "s"(limit)
        : "vcc");
    return m;
}

// Staged positions of a set, two at a time: x0 x1 y0 y1 z0 z1.  Four positions
// are 48 consecutive bytes, three reads at one address.
struct PosStage {
    float d[3 * kNbrStage + 12];   // the candidate tests read up to three positions past a range
    __device__ __forceinline__ void put(uint32_t k, const float4& p)
    {
        float* q = d + 6u * (k >> 1) + (k & 1u);
        q[0] = p.x; q[2] = p.y; q[4] = p.z;
    }
};

// Which of the staged positions [l0, min(l0 + 32, e)) lie within the support of
// p: bit k for l0 + k.  l0 is even; each step tests four positions, 8 vector
// instructions a candidate.  The last step may test up to three positions past
// e, whose bits are cleared.
__device__ __forceinline__ uint32_t near_mask(const PosStage& st, const float4& p, float hk2, uint32_t l0, uint32_t e)
{
    typedef float f4 __attribute__((ext_vector_type(4), aligned(8)));
    const uint32_t cnt = min(e - l0, 32u);
    uint32_t m = 0, t = 3u * l0;                         // in words
    const uint32_t end = t + 3u * cnt;
#pragma unroll 1
    do {
        const f4 a = *reinterpret_cast<const f4*>(st.d + t), b = *reinterpret_cast<const f4*>(st.d + t + 4),
                 c = *reinterpret_cast<const f4*>(st.d + t + 8);
        m = shift_in_less(m, dist2(p.x - a[0], p.y - a[2], p.z - b[0]), dist2(p.x - a[1], p.y - a[3], p.z - b[1]),
                          dist2(p.x - b[2], p.y - c[0], p.z - c[2]), dist2(p.x - b[3], p.y - c[1], p.z - c[3]), hk2);
        t += 12u;
    } while (t < end);
    // (cnt + 3) / 4 steps made, the first candidate in the highest of their bits
    m = __builtin_bitreverse32(m) >> ((32u - cnt) & ~3u);
    return cnt < 32u ? m & ((1u << cnt) - 1u) : m;
}

// the lowest `count` set bits of m (count < popc(m))
__device__ __forceinline__ uint32_t lowest_bits(uint32_t m, uint32_t count)
{
    uint32_t r = 0;
    for (; count > 0u; --count) { r |= m & (0u - m); m &= m - 1u; }
    return r;
}

// visit(q, position of at(q)) for q in [s0, e), four positions loaded at a time (eight do
// not fit 64 registers): the search of blocks without tables or 16-bit
// lists is one lane's chain of reads.  REST: what is left of a range singly.  Cells hold
// 8 to 12 particles, and a masked batch wastes up to three tests of each, which the
// few blocks that outlast a sorted search do not feel (the sparsest spray 69 us, with the rest singly 70),
// but an unsorted search does, where every block reads so: 150k particles
// 177 us masked, 139 with the rest singly, 1.05 M 552 and 463.
constexpr uint32_t kScanBatch = 4;
template <bool REST, class At, class Visit>
__device__ __forceinline__ void scan_positions(const float4* __restrict__ pos, uint32_t s0, uint32_t e, At&& at, Visit&& visit)
{
    uint32_t q = s0;
#pragma unroll 1
    for (; REST ? q + kScanBatch <= e : q < e; q += kScanBatch) {
        float4 t[kScanBatch];
#pragma unroll
        for (uint32_t u = 0; u < kScanBatch; ++u) t[u] = pos[at(REST ? q + u : min(q + u, e - 1u))];
#pragma unroll
        for (uint32_t u = 0; u < kScanBatch; ++u)
            if (REST || q + u < e) visit(q + u, t[u]);
    }
    if (REST) {
#pragma unroll 1
        for (; q < e; ++q) visit(q, pos[at(q)]);
    }
}

// DFSPH_neighborsSearch_kernel<true> (DFSPH_core_cuda.cu:2219-2531,
// DFSPH_macro_cuda.h:136-155): every fluid particle within h (strict, FP32) of
// particle i except i itself, over the 27 cells around its cell, then the
// boundary particles the same way, at most max_neighbors in total (fluid
// first).  Cells are visited in for_each_adjacent_cell's order (y, then z,
// then x) and each cell's particles in index order, in every list form.
//
// Each block also builds its neighbor set: the set cells are marked in the
// row masks, numbered by a block scan over the rows, and get their fluid
// ranges, set offsets and boundary ranges, one thread per cell.  Every lane then
// keeps its 9 rows as (first, last) set cells in registers.  The set's positions
// are staged in LDS for the candidate tests (over the masks, which are dead by
// then), with the boundary's behind them where both fit.  Sets up to kStageCap
// store 16-bit lists; larger ones, blocks whose tables do not fit, and the INDIRECT search (fluid
// not reordered, the grid indexes it through perm: the need_sort == false
// path) store 32-bit global lists.
//
// What bounds it: vector instructions (2.7e8 a search of 4.19 M particles, the
// rate of all SIMDs), over half of them in near_mask's loop and a quarter in
// the list writers, whose loops run for the wave's longest lane.  64 VGPRs and
// 40 KB keep four blocks per CU.  Against the version with a dense cell table,
// binary searches for the stage and 16-byte position records: 597 -> 416 us
// (4.19 M particles, spacing 2r), one block's walls 15 -> 8 us, and blocks of
// spray have tables (1 M dam break, 40 steps: 11 -> 5 blocks without).
template <bool INDIRECT>
__global__ __launch_bounds__(kBlock, DFSPH_BLOCK == 512 ? 8 : 4) void k_neighbors(SimConst c, const float4* __restrict__ pos,
                                                      const uint32_t* __restrict__ cs_f,
                                                      const uint32_t* __restrict__ perm,
                                                      const float4* __restrict__ bpos,
                                                      const uint32_t* __restrict__ cs_b, uint32_t n,
                                                      uint16_t* __restrict__ nbr16, uint32_t* __restrict__ nbrf,
                                                      uint32_t* __restrict__ nbrb, uint32_t* __restrict__ cnt,
                                                      uint32_t* __restrict__ stage_n, uint32_t* __restrict__ stg,
                                                      Restrict rs, uint4* __restrict__ part, uint32_t split)
{
    // The tables under construction lie in the first half of the staged
    // positions and are dead once those are loaded.
    __shared__ __align__(16) PosStage st;
    unsigned long long* s_mask = reinterpret_cast<unsigned long long*>(st.d);   // x positions of the row's set cells
    uint32_t* s_place = reinterpret_cast<uint32_t*>(s_mask + kSetRows);   // box places of the set cells
    uint16_t* s_first = reinterpret_cast<uint16_t*>(s_place + kSetCells); // number of the row's first set cell
    static_assert(kSetRows * 10 + kSetCells * 4 <= kHalfStage * 12 && kSetRows * 8 + kBigCells * 4 <= kHalfStage * 12,
                  "tables under construction exceed half the stage");
    // four words per set cell (one more for the offsets): set offset of its fluid
    // particles and what to add for their indices, the same for its boundary ones
    __shared__ uint32_t s_tab[4 * kSetCells + 2];
    static_assert(4 * kSetCells + 2 >= kBigCells + 1 + kSetRows / 2,
                  "the boundary offsets of a large table and its rows' first cells lie in s_tab");
    uint32_t *s_off = s_tab, *s_src = s_tab + kSetCells + 1, *s_boff = s_src + kSetCells, *s_bs = s_boff + kSetCells + 1;
    constexpr int NW = kBlock / 64;
    __shared__ int s_w[6 * NW];
    static_assert((kStageCap - 1) * 16 <= 0xffffu && kBigCells < 0xffffu, "16-bit byte offsets / cell ids");
    uint32_t* s_wu = reinterpret_cast<uint32_t*>(s_w);

    // split blocks build the same set, each searches its share of the wavefronts
    const uint32_t b = xcd_block() / split, share = xcd_block() % split;
    const uint32_t i = b * kBlock + threadIdx.x;
    const bool act = i < n;
    const bool mine = (threadIdx.x >> 6) / (kBlock / 64u / split) == share;
    float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    int cx = 0, cy = 0, cz = 0;
    if (act) {
        p = pos[i];
        cx = cell_coord(c, p.x, 0);
        cy = cell_coord(c, p.y, 1);
        cz = cell_coord(c, p.z, 2);
    }
    uint32_t S = kUnstaged, U = 0, uown = 0, Sb = 0;
    uint32_t row[9];
#pragma unroll
    for (int r = 0; r < 9; ++r) row[r] = kNoRow;
    bool tabled = false;                        // block uniform: row / s_off / s_src / s_b* valid
    if (!INDIRECT && n <= b * kBlock) S = 0;    // a block past the end: empty set
    if (!INDIRECT && n > b * kBlock) {
        // bounding box of the set cells, clamped to the grid
        const int w = threadIdx.x >> 6;
        const int lo_x = wave_min_i(act ? cx : kIntMax), hi_x = wave_max_i(act ? cx : -1);
        const int lo_y = wave_min_i(act ? cy : kIntMax), hi_y = wave_max_i(act ? cy : -1);
        const int lo_z = wave_min_i(act ? cz : kIntMax), hi_z = wave_max_i(act ? cz : -1);
        if ((threadIdx.x & 63) == 0) {
            s_w[w] = lo_x; s_w[NW + w] = lo_y; s_w[2 * NW + w] = lo_z;
            s_w[3 * NW + w] = hi_x; s_w[4 * NW + w] = hi_y; s_w[5 * NW + w] = hi_z;
        }
        for (uint32_t k = threadIdx.x; k < kSetRows / 2; k += kBlock)
            reinterpret_cast<uint4*>(s_mask)[k] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        int lo[3] = {kIntMax, kIntMax, kIntMax}, hi[3] = {-1, -1, -1};
#pragma unroll
        for (int k = 0; k < NW; ++k) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                lo[a] = min(lo[a], s_w[NW * a + k]);
                hi[a] = max(hi[a], s_w[NW * (3 + a) + k]);
            }
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = max(__builtin_amdgcn_readfirstlane(lo[a]) - 1, 0);
            hi[a] = min(__builtin_amdgcn_readfirstlane(hi[a]) + 1, c.dim[a] - 1);
        }
        const uint32_t W = (uint32_t)(hi[0] - lo[0] + 1), D = (uint32_t)(hi[2] - lo[2] + 1), H = (uint32_t)(hi[1] - lo[1] + 1);
        const bool fits = W <= kBoxW && D <= kBoxD && H <= kSetRows && D * H <= kSetRows;
        const uint32_t R = D * H;
        const int xl = max(cx - 1, 0), xh = min(cx + 1, c.dim[0] - 1);
        const uint32_t bx = (uint32_t)(xl - lo[0]);                                // first x of my rows, in the box
        const uint32_t nx = (uint32_t)(xh - xl);
        const uint32_t own = (uint32_t)(cz - lo[2]) + D * (uint32_t)(cy - lo[1]);
        if (fits) {
            // mark the 27 cells, one lane per run of a cell in a wave
            const uint32_t lin = act ? (uint32_t)(cx - lo[0]) + W * own : kKeyInvalid;
            const uint32_t prev = (uint32_t)__builtin_amdgcn_update_dpp((int)kKeyInvalid, (int)lin, 0x138, 0xf, 0xf, false);
            if (act && ((threadIdx.x & 63) == 0 || prev != lin)) {
                const unsigned long long bits = ((2ull << nx) - 1ull) << bx;
#pragma unroll
                for (int r = 0; r < 9; ++r) {
                    const int y = cy + r / 3 - 1, z = cz + r % 3 - 1;
                    if (y >= 0 && y < c.dim[1] && z >= 0 && z < c.dim[2])
                        atomicOr(&s_mask[own + (uint32_t)(r % 3 - 1) + D * (uint32_t)(r / 3 - 1)], bits);
                }
            }
        }
        // The masks are complete and the boxes in s_w are read: its words are
        // used again by the scans, or, of a block that does not fit, by the statistics.
        __syncthreads();
        if (fits) {
            // number the marked cells row by row; thread t owns rows [tE, tE + E)
            const uint32_t E = (R + kBlock - 1) / kBlock;
            const uint32_t k0 = threadIdx.x * E, k1 = min(k0 + E, R);
            uint32_t occ = 0;
            for (uint32_t k = k0; k < k1; ++k) occ += (uint32_t)__popcll(s_mask[k]);
            uint32_t ubase = 0;
            U = (uint32_t)__builtin_amdgcn_readfirstlane((int)block_excl_scan_u(occ, &ubase, s_wu));
            const bool big = U > kSetCells;
            tabled = U <= kBigCells;
            if (big) {
                s_off = reinterpret_cast<uint32_t*>(st.d + 3 * kHalfStage);
                s_src = s_off + kHalfStage;
                s_bs = s_src + kHalfStage;
                s_boff = s_tab;
                s_first = reinterpret_cast<uint16_t*>(s_tab + kBigCells + 1);
            }
            if (tabled) {
                for (uint32_t k = k0; k < k1; ++k) {
                    const uint32_t y = k / D, at = ((k - y * D) << kPlaceZ) | (y << kPlaceY);
                    s_first[k] = (uint16_t)ubase;
                    for (unsigned long long m = s_mask[k]; m != 0ull; m &= m - 1ull)
                        s_place[ubase++] = at | (uint32_t)(__ffsll((long long)m) - 1);
                }
                __syncthreads();
                // fluid and boundary ranges of the set cells, thread t's being [tC, tC + C)
                constexpr uint32_t CMAX = (kBigCells + kBlock - 1) / kBlock;
                const uint32_t C = U <= (uint32_t)kBlock ? 1u : CMAX;
                uint32_t cf[CMAX], cb[CMAX], f0s[CMAX], b0s[CMAX], fsum = 0, bsum = 0;
#pragma unroll
                for (uint32_t k = 0; k < CMAX; ++k) {
                    const uint32_t u = threadIdx.x * C + k;
                    cf[k] = cb[k] = f0s[k] = b0s[k] = 0u;
                    if (k < C && u < U) {
                        const uint32_t at = s_place[u];
                        const uint32_t key = cell_key(c, lo[0] + (int)(at & (kBoxW - 1u)), lo[1] + (int)(at >> kPlaceY),
                                                      lo[2] + (int)((at >> kPlaceZ) & (kBoxD - 1u)));
                        const uint32_t f0 = cs_f[key], f1 = cs_f[key + 1], b0 = cs_b[key], b1 = cs_b[key + 1];
                        f0s[k] = f0;
                        b0s[k] = b0;
                        cf[k] = f1 - f0;
                        cb[k] = b1 - b0;
                    }
                    fsum += cf[k];
                    bsum += cb[k];
                }
                // both exclusive scans between one pair of barriers
                const uint32_t fi = wave_incl_scan_u(fsum), bi = wave_incl_scan_u(bsum);
                if ((threadIdx.x & 63) == 63) { s_wu[w] = fi; s_wu[NW + w] = bi; }
                __syncthreads();
                uint32_t foff = fi - fsum, boff = bi - bsum, tot = 0;
#pragma unroll
                for (int k = 0; k < NW; ++k) {
                    foff += k < w ? s_wu[k] : 0u;
                    boff += k < w ? s_wu[NW + k] : 0u;
                    tot += s_wu[k];
                    Sb += s_wu[NW + k];
                }
                tot = (uint32_t)__builtin_amdgcn_readfirstlane((int)tot);
                Sb = (uint32_t)__builtin_amdgcn_readfirstlane((int)Sb);
#pragma unroll
                for (uint32_t k = 0; k < CMAX; ++k) {
                    const uint32_t u = threadIdx.x * C + k;
                    if (k < C && u < U) {
                        s_off[u] = foff;
                        s_boff[u] = boff;
                        s_src[u] = f0s[k] - foff;
                        s_bs[u] = b0s[k] - boff;
                    }
                    foff += cf[k];
                    boff += cb[k];
                }
                if (threadIdx.x == 0) { s_off[U] = tot; s_boff[U] = Sb; }
                S = tot <= c.stage_cap ? tot : kUnstaged;
                // each lane's rows (dy, dz) as (first, last) set cell of x-1..x+1
                if (act && mine) {
#pragma unroll
                    for (int r = 0; r < 9; ++r) {
                        const int y = cy + r / 3 - 1, z = cz + r % 3 - 1;
                        if (y >= 0 && y < c.dim[1] && z >= 0 && z < c.dim[2]) {
                            const uint32_t k = own + (uint32_t)(r % 3 - 1) + D * (uint32_t)(r / 3 - 1);
                            const uint32_t u = s_first[k] + (uint32_t)__popcll(s_mask[k] & ((1ull << bx) - 1ull));
                            row[r] = u | ((u + nx) << 16);
                            if (r == 4) uown = u + (uint32_t)(cx - xl);
                        }
                    }
                }
                __syncthreads();                // the table area is staged over next
            }
        }
    }
    const uint32_t room = U <= kSetCells ? kNbrStage : kHalfStage;
    const bool lds_search = S <= room && c.stage_lds > 0u;
    const bool lds_bnd = lds_search && S + Sb <= room;        // boundary staged at [S, S + Sb)
    if (threadIdx.x == 0 && share == 0u) stage_n[b] = S == kUnstaged || S <= c.stage_lds ? S : (S | kSetNoLds);
    if (S != kUnstaged) {
        // eight lanes per set cell: its particles' ids and positions to their set places
        uint32_t* g_out = stg + (size_t)b * kStageCap;
        const uint32_t sub = threadIdx.x & 7u;
        for (uint32_t u = threadIdx.x >> 3; u < U; u += kBlock / 8) {
            const uint32_t off = s_off[u], e = s_off[u + 1u], g0 = s_src[u];
            for (uint32_t k = off + sub; k < e; k += 8u) {
                if (lds_search) st.put(k, pos[g0 + k]);
                if (share == 0u) g_out[k] = g0 + k;
            }
            if (lds_bnd) {
                const uint32_t boff = s_boff[u], be = s_boff[u + 1u], j0 = s_bs[u];
                for (uint32_t k = boff + sub; k < be; k += 8u) st.put(S + k, bpos[j0 + k]);
            }
        }
        __syncthreads();
    }
    const bool searches = act && mine && is_source(rs, i);
    if (act && mine && !searches) cnt[i] = 0;   // restricted out: no lists
    const uint32_t maxn = c.max_nbr, cap = c.cap;
    const float hk2 = c.hk2;
    uint32_t nf = 0, nb = 0;                     // found; stored while below max_neighbors
    // Each row range goes in chunks of up to 32 candidates: a branch-free pass
    // sets one bit per candidate within h, then the set bits are appended in
    // order.  [s0, e): the range in the stage, which holds the set from w0 on.
    auto fluid_range = [&](ListWriter16& w, uint32_t self, uint32_t s0, uint32_t e, uint32_t w0) {
        for (uint32_t l0 = s0 & ~1u; l0 < e; l0 += 32u) {
            uint32_t m = near_mask(st, p, hk2, l0, e);
            if (l0 < s0) m &= ~1u;               // the position before the range
            if (self - w0 - l0 < 32u) m &= ~(1u << (self - w0 - l0));
            const uint32_t hits = (uint32_t)__popc(m);
            if (nf + hits > maxn) m = lowest_bits(m, nf < maxn ? maxn - nf : 0u);
            nf += hits;
            for (; m != 0u; m &= m - 1u) w.push((w0 + l0 + (uint32_t)__builtin_ctz(m)) << 4);   // LDS byte offset
        }
    };
    if (S != kUnstaged && !lds_search) {
        // Sets beyond the stage pass through it in windows, each lane's rows cut
        // to the window; the set's order is the rows' order, so the lists
        // are the same.  With the walls below, against four global reads at a time:
        // the wave tank's search (260k) 81 -> 66 us, 258k particles with walls at
        // spacing r 142 -> 128, 200k with spray 95 -> 85 (4.19 M: 438 -> 442).
        ListWriter16 w{reinterpret_cast<uint4*>(nbr16) + i, cap};
        const uint32_t self = searches ? i - s_src[uown] : 0u;
        for (uint32_t w0 = 0; w0 < S; w0 += room) {
            const uint32_t w1 = min(w0 + room, S);
            __syncthreads();                     // the window before is read
            for (uint32_t u = threadIdx.x >> 3; u < U; u += kBlock / 8) {
                const uint32_t e = min(s_off[u + 1u], w1), g0 = s_src[u];
                for (uint32_t k = max(s_off[u], w0) + (threadIdx.x & 7u); k < e; k += 8u) st.put(k - w0, pos[g0 + k]);
            }
            __syncthreads();
#pragma unroll 1
            for (int r = 0; r < 9; ++r) {
                if (!searches || row[r] == kNoRow) continue;
                const uint32_t s0 = max(s_off[row[r] & 0xffffu], w0), e = min(s_off[(row[r] >> 16) + 1u], w1);
                if (s0 < e) fluid_range(w, self, s0 - w0, e - w0, w0);
            }
        }
        if (searches) w.finish();
    } else if (searches) {
        if (S != kUnstaged) {
            ListWriter16 w{reinterpret_cast<uint4*>(nbr16) + i, cap};
            const uint32_t self = i - s_src[uown];
#pragma unroll 1
            for (int r = 0; r < 9; ++r) {
                if (row[r] == kNoRow) continue;
                fluid_range(w, self, s_off[row[r] & 0xffffu], s_off[(row[r] >> 16) + 1u], 0u);
            }
            w.finish();
        } else {
            ListWriter32 w{reinterpret_cast<uint4*>(nbrf) + i, cap};
            auto scan_range = [&](uint32_t s0, uint32_t e) {
                auto index = [&](uint32_t q) { return INDIRECT ? perm[q] : q; };
                scan_positions<INDIRECT>(pos, s0, e, index, [&](uint32_t q, const float4& pj) {
                    if (dist2(p.x - pj.x, p.y - pj.y, p.z - pj.z) < hk2) {
                        const uint32_t j = index(q);
                        if (j != i) {
                            if (nf < maxn) w.push(j);
                            ++nf;
                        }
                    }
                });
            };
            if (tabled) {
#pragma unroll 1
                for (int r = 0; r < 9; ++r) {
                    if (row[r] == kNoRow) continue;
                    for (uint32_t u = row[r] & 0xffffu; u <= (row[r] >> 16); ++u)
                        scan_range(s_src[u] + s_off[u], s_src[u] + s_off[u + 1u]);
                }
            } else {
                for_each_adjacent_range(c, cx, cy, cz, cs_f, scan_range);
            }
            w.finish();
        }
    }
    const uint32_t sf = nf < maxn ? nf : maxn;
    ListWriter32 wb{reinterpret_cast<uint4*>(nbrb) + i, cap};
    // A row's boundary particles are one contiguous staged range, in up to
    // three runs of boundary indices (one per cell).  at: what the stage begins
    // with; [w0, w1): the boundary offsets that follow it.
    auto boundary_row = [&](uint32_t rw, uint32_t at, uint32_t w0, uint32_t w1) {
        const uint32_t u0 = rw & 0xffffu, u1 = rw >> 16;
        const uint32_t b0 = max(s_boff[u0], w0), b1 = min(s_boff[u1 + 1u], w1);
        if (b0 >= b1) return;
        const uint32_t mv = at - w0, s0 = b0 + mv, e = b1 + mv;
        const uint32_t ub = min(u0 + 1u, u1), k1 = s_boff[ub] + mv, k2 = s_boff[u1] + mv;
        const uint32_t j0 = s_bs[u0] - mv, j1 = s_bs[ub] - mv, j2 = s_bs[u1] - mv;
        for (uint32_t l0 = s0 & ~1u; l0 < e; l0 += 32u) {
            uint32_t m = near_mask(st, p, hk2, l0, e);
            if (l0 < s0) m &= ~1u;               // the position before the range
            const uint32_t hits = (uint32_t)__popc(m);
            if (sf + nb + hits > maxn) m = lowest_bits(m, sf + nb < maxn ? maxn - sf - nb : 0u);
            nb += hits;
            for (; m != 0u; m &= m - 1u) {
                const uint32_t k = l0 + (uint32_t)__builtin_ctz(m);
                wb.push(k + ((int)(k - k1) < 0 ? j0 : (int)(k - k2) < 0 ? j1 : j2));
            }
        }
    };
    if (lds_bnd) {
        if (Sb > 0u && searches) {
#pragma unroll 1
            for (int r = 0; r < 9; ++r)
                if (row[r] != kNoRow) boundary_row(row[r], S, 0u, Sb);
        }
    } else if (tabled) {
        // the walls after the fluid, in windows of the stage
        for (uint32_t w0 = 0; w0 < Sb; w0 += room) {
            const uint32_t w1 = min(w0 + room, Sb);
            __syncthreads();                     // the stage's last contents are read
            for (uint32_t u = threadIdx.x >> 3; u < U; u += kBlock / 8) {
                const uint32_t e = min(s_boff[u + 1u], w1), j0 = s_bs[u];
                for (uint32_t k = max(s_boff[u], w0) + (threadIdx.x & 7u); k < e; k += 8u) st.put(k - w0, bpos[j0 + k]);
            }
            __syncthreads();
#pragma unroll 1
            for (int r = 0; r < 9; ++r)
                if (searches && row[r] != kNoRow) boundary_row(row[r], 0u, w0, w1);
        }
    } else if (searches) {
        for_each_adjacent_range(c, cx, cy, cz, cs_b, [&](uint32_t s0, uint32_t e) {
            scan_positions<INDIRECT>(bpos, s0, e, [](uint32_t j) { return j; }, [&](uint32_t j, const float4& pj) {
                if (dist2(p.x - pj.x, p.y - pj.y, p.z - pj.z) < hk2) {
                    if (sf + nb < maxn) wb.push(j);
                    ++nb;
                }
            });
        });
    }
    uint32_t total = 0, trunc = 0, stored_f = 0, stored_b = 0, stored_u32 = 0;
    if (searches) {
        const uint32_t sb = nb < maxn - sf ? nb : maxn - sf;
        wb.finish();
        total = nf + nb;
        trunc = total > maxn ? 1u : 0u;
        cnt[i] = sf | (sb << 16);
        stored_f = sf;
        stored_b = sb;
        stored_u32 = S == kUnstaged ? sf : 0u;
    }
    // the block's statistics go to its two records in part (k_nbr_finalize
    // sums them): per-wave atomics on one control line would serialise
    const uint32_t wv[5] = {(uint32_t)wave_max_i((int)total), wave_total_u(trunc), wave_total_u(stored_f),
                            wave_total_u(stored_b), wave_total_u(stored_u32)};
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 5; ++k) s_w[5 * w + k] = (int)wv[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t a[5] = {0u, 0u, 0u, 0u, 0u};
        for (int v = 0; v < NW; ++v)
            for (int k = 0; k < 5; ++k) {
                const uint32_t x = (uint32_t)s_w[5 * v + k];
                a[k] = k == 0 ? max(a[0], x) : a[k] + x;
            }
        const uint32_t unstaged = S > c.stage_lds && n > b * kBlock && share == 0u ? 1u : 0u;
        part[2 * xcd_block()] = make_uint4(a[0], a[1], a[2], a[3]);
        part[2 * xcd_block() + 1] = make_uint4(a[4], unstaged, 0u, 0u);
    }
}

// The neighbor statistics of the last search from the block records of
// k_neighbors (maximum, sums in a fixed order).
__global__ __launch_bounds__(kBlock) void k_nbr_finalize(const uint4* __restrict__ part, uint32_t nblocks, DevCtl* ctl)
{
    __shared__ unsigned long long s[6][kBlock];
    unsigned long long a[6] = {0, 0, 0, 0, 0, 0};
    for (uint32_t b = threadIdx.x; b < nblocks; b += kBlock) {
        const uint4 p = part[2 * b], q = part[2 * b + 1];
        a[0] = a[0] > p.x ? a[0] : p.x;
        a[1] += p.y; a[2] += p.z; a[3] += p.w; a[4] += q.x; a[5] += q.y;
    }
    for (int k = 0; k < 6; ++k) s[k][threadIdx.x] = a[k];
    __syncthreads();
    for (uint32_t h = kBlock / 2; h > 0; h >>= 1) {
        if (threadIdx.x < h)
            for (int k = 0; k < 6; ++k) {
                const unsigned long long o = s[k][threadIdx.x + h];
                s[k][threadIdx.x] = k == 0 ? (s[0][threadIdx.x] > o ? s[0][threadIdx.x] : o) : s[k][threadIdx.x] + o;
            }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        ctl->max_seen = (uint32_t)s[0][0];
        ctl->overflow = (uint32_t)s[1][0];
        ctl->nbr_fluid = s[2][0];
        ctl->nbr_boundary = s[3][0];
        ctl->nbr_fluid_unstaged = s[4][0];
        ctl->unstaged_blocks = (uint32_t)s[5][0];
    }
}

// Every list of the last search as 32-bit global ids, fluid then boundary
// (the reference's plain interleaved layout, slot k at k * cap + i), for readback.
__global__ __launch_bounds__(kBlock) void k_expand_lists(uint32_t n, uint32_t cap, NbrLists L, uint32_t* out)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t b = i / kBlock;
    const uint32_t cn = L.cnt[i];
    const uint32_t nf = cn & 0xffffu, nb = cn >> 16;
    const uint32_t sn = L.stage_n[b];
    for (uint32_t k = 0; k < nf; ++k) {
        uint32_t j;
        if (sn != kUnstaged) {
            const uint32_t l = L.nbr16[(((size_t)(k >> 3) * cap + i) << 3) + (k & 7u)] >> 4;
            j = L.stg[(size_t)b * kStageCap + l];
        } else {
            j = L.nbrf[(((size_t)(k >> 2) * cap + i) << 2) + (k & 3u)];
        }
        out[(size_t)k * cap + i] = j;
    }
    for (uint32_t k = 0; k < nb; ++k)
        out[(size_t)(nf + k) * cap + i] = L.nbrb[(((size_t)(k >> 2) * cap + i) << 2) + (k & 3u)];
}

// FluidModel::computeBoundaryPsi (FluidModel.cpp:233-258) on the device:
// psi_i = rho0 / (W0 + sum_{j != i, |xij| < h} W(xij)) over the boundary set.
__global__ void k_boundary_psi(SimConst c, const float4* bpos, const uint32_t* cs_b, uint32_t nb, float* psi)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nb) return;
    const float4 p = bpos[i];
    const int cx = cell_coord(c, p.x, 0), cy = cell_coord(c, p.y, 1), cz = cell_coord(c, p.z, 2);
    float delta = c.W0;
    for_each_adjacent_cell(c, cx, cy, cz, [&](uint32_t nk) {
        for (uint32_t j = cs_b[nk]; j < cs_b[nk + 1]; ++j) {
            if (j == i) continue;
            const float4 q = bpos[j];
            const float r2 = dist2(p.x - q.x, p.y - q.y, p.z - q.z);
            if (r2 < c.hk2) delta += kernel_W(c, r2);
        }
    });
    psi[i] = c.density0 / delta;
}

__global__ void k_set_w(float4* p, const float* w, uint32_t n)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i].w = w[i];
}

// ------------------------------------------------------------------------
// solver sweeps
// ------------------------------------------------------------------------

// neighbor records loaded in the first phase of a batch
struct PV {
    float4 p, v;                   // position + mass, velocity (+ a per-kernel scalar in w)
};

// LDS stage of (position, velocity) records.  UM (every fluid particle has the
// mass c.m_uniform): 24 B per particle, (x y z vx) and (vy vz), so that two
// 512-particle blocks fit a CU (78 KB each) instead of one; the mass is put
// back from the constant, the same value bit for bit.  Entries of the 16-bit
// lists are byte offsets of 16-byte slots; the 8-byte slots are at half.
template <bool UM>
struct PVStage {
    float4 p[kStageMaxPV], v[kStageMaxPV];
    __device__ __forceinline__ void put(uint32_t k, const PV& d) { p[k] = d.p; v[k] = d.v; }
    __device__ __forceinline__ PV get(uint32_t off, float) const { return PV{lds_f4(p, off), lds_f4(v, off)}; }
};
template <>
struct PVStage<true> {
    float4 a[kStageMaxPV];
    float2 b[kStageMaxPV];
    __device__ __forceinline__ void put(uint32_t k, const PV& d)
    {
        a[k] = make_float4(d.p.x, d.p.y, d.p.z, d.v.x);
        b[k] = make_float2(d.v.y, d.v.z);
    }
    __device__ __forceinline__ PV get(uint32_t off, float m) const
    {
        const float4 u = lds_f4(a, off);
        const float2 w = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(b) + (off >> 1));
        return PV{make_float4(u.x, u.y, u.z, m), make_float4(u.w, w.x, w.y, 0.0f)};
    }
};
// LDS stage of (position, velocity, scalar) records.  UM: 28 B per particle,
// (x y z vx), (vy vz) and the scalar, the mass put back from the constant;
// otherwise 32 B, (x y z m) and (vx vy vz scalar).
template <bool UM>
struct PVSStage {
    float4 p[kStageMaxX], v[kStageMaxX];
    __device__ __forceinline__ void put(uint32_t k, const PV& d) { p[k] = d.p; v[k] = d.v; }
    __device__ __forceinline__ PV get(uint32_t off, float) const { return PV{lds_f4(p, off), lds_f4(v, off)}; }
};
template <>
struct PVSStage<true> {
    float4 a[kStageMaxX];
    float2 b[kStageMaxX];
    float s[kStageMaxX];
    __device__ __forceinline__ void put(uint32_t k, const PV& d)
    {
        a[k] = make_float4(d.p.x, d.p.y, d.p.z, d.v.x);
        b[k] = make_float2(d.v.y, d.v.z);
        s[k] = d.v.w;
    }
    __device__ __forceinline__ PV get(uint32_t off, float m) const
    {
        const float4 u = lds_f4(a, off);
        const float2 w = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(b) + (off >> 1));
        const float q = lds_f1(s, off);
        return PV{make_float4(u.x, u.y, u.z, m), make_float4(u.w, w.x, w.y, q)};
    }
};

struct PK {
    float4 p;                      // position + mass
    float k;                       // k_j of the Jacobi sweep / the warm start
};

// LDS stage of (position, k) records: 20 B per particle, or 16 B (x y z k)
// with a uniform fluid mass (UM; three 512-particle blocks per CU instead of
// two).
template <bool UM>
struct PKStage {
    float4 p[kStageMax];
    float k[kStageMax];
    __device__ __forceinline__ void put(uint32_t i, const PK& d) { p[i] = d.p; k[i] = d.k; }
    __device__ __forceinline__ PK get(uint32_t off, float) const { return PK{lds_f4(p, off), lds_f1(k, off)}; }
};
template <>
struct PKStage<true> {
    float4 a[kStageMax];
    __device__ __forceinline__ void put(uint32_t i, const PK& d) { a[i] = make_float4(d.p.x, d.p.y, d.p.z, d.k); }
    __device__ __forceinline__ PK get(uint32_t off, float m) const
    {
        const float4 u = lds_f4(a, off);
        return PK{make_float4(u.x, u.y, u.z, m), u.w};
    }
};

// Reducing sweeps write one FP64 partial per block with a plain store; the
// separate one-block kernel below sums them.  (A "last block finishes"
// reduction inside the sweep needs a device-scope release/acquire per block,
// which on MI355X writes back and invalidates the XCD's L2 every time and
// throws away the neighbor data the other blocks are gathering.)
__device__ __forceinline__ void store_partial(double* partial, double bsum)
{
    if (threadIdx.x == 0) partial[blockIdx.x] = bsum;
}

// Sums the block partials in a fixed order (deterministic), forms
// err = sum / N and evaluates the loop condition of cuda_divergenceSolve /
// cuda_pressureSolve: continue while ((err > eta) || (it < min)) && (it < max).
// it: the iterations made.  Below the minimum the loop continues whatever the
// error, so only the iterations from the minimum on are followed by this kernel
// (a launch and a one-block kernel, 4 to 6 us, three times less a step).
__global__ __launch_bounds__(kBlock) void k_solve_finalize(SolveCtl* ctl, const double* partial, uint32_t nparts,
                                                          uint32_t it, Publish pub)
{
    __shared__ double lds4[kBlock / 64];
    if (!ctl->done) {
        // each thread sums its strided share in order; the loads of 8 terms
        // are issued together (adding the 0.0 of a missing term is exact, so
        // the sum is the one-at-a-time sum, bit for bit)
        constexpr uint32_t kBatch = 8;
        double acc = 0.0;
        for (uint32_t k0 = threadIdx.x; k0 < nparts; k0 += kBatch * kBlock) {
            double v[kBatch];
#pragma unroll
            for (uint32_t u = 0; u < kBatch; ++u) {
                const uint32_t k = k0 + u * kBlock;
                v[u] = k < nparts ? partial[k] : 0.0;
            }
#pragma unroll
            for (uint32_t u = 0; u < kBatch; ++u) acc += v[u];
        }
        const double tot = block_sum(acc, lds4);
        if (threadIdx.x == 0) {
            const double err = ctl->n_div > 0.0 ? tot / ctl->n_div : 0.0;
            ctl->sum = tot;
            ctl->err = err;
            ctl->iters = it;
            const bool cont = ((err > ctl->eta) || (it < ctl->min_iter)) && (it < ctl->max_iter);
            ctl->done = cont ? 0u : 1u;
        }
    }
    if (threadIdx.x == 0 && pub.rec) publish(pub, ctl);
}

// Fused density + factor + divergence source, then the divergence warm start:
// DFSPH_divergence_warmstart_init_kernel (DFSPH_core_cuda.cu:220-376) followed by
// DFSPH_divergence_compute_kernel<true> (:495-517, divergenceSolveParticle :400-481).
// rho_i = m_i W0 + sum m_j W_ij; alpha_i = -(1/h) / max(sum |m_j gradW|^2 + |sum m_j gradW|^2, eps);
// rho_adv_i = 0 if fewer than 20 neighbors else max(sum m_j (v_i - v_j).gradW, 0).
// Warm start (only where rho_adv_i > 0): v_i += h sum (k_i + k_j) m_j gradW with
// k = max(kappaV h_ratio / 2, -0.5) (WS == 0), that value plus the learned
// correction, bounded by ws_learned with half the last converged total
// (WS == 1), or nothing (WS == 2).  kws holds
// the last solve's kappaV increments.  Velocities are read from vel_i and
// written to vel_o.  The applied k_i starts the particle's total of the step
// in kvtot (when given).
// <0, true, true> (bodies) is two registers over the 128 of two blocks per CU and
// keeps an address in scratch across the loop over 32-bit lists; with the own mass
// from the constants it fits, but takes 33.5 us instead of 33.1 in the wave tank (260k).
template <int WS, bool SOL, bool UM>
__global__ __launch_bounds__(kBlock, UM ? DFSPH_PV_WAVES : 1) void k_div_ws_init(SimConst c, const DevTime* t, uint32_t n,
                                                        const float4* __restrict__ pos,
                                                        const float4* __restrict__ bpos, NbrLists L,
                                                        const float4* __restrict__ vel_i,
                                                        float4* __restrict__ vel_o,
                                                        const float* __restrict__ kws, WsLearned lw,
                                                        float* __restrict__ rho, float* __restrict__ alpha,
                                                        float* __restrict__ radv, float* __restrict__ kvtot)
{
    __shared__ PVSStage<UM> st;                  // (x, v, warm-start k) of the staged set
    const float ratio = t->ratio, h = t->h, inv_h = t->inv_h;
    auto ws_of = [&](uint32_t j) -> float {
        if (WS == 2) return 0.0f;
        const float ref = fmaxf(kws[j] * ratio / 2.0f, -0.5f);
        if (WS == 0) return ref;
        return ws_learned(ref, fmaxf(0.5f * lw.prev[j] * inv_h, -0.5f), lw.dy[j] * lw.scale * inv_h);
    };
    const uint32_t b = xcd_block();
    const uint32_t i = b * kBlock + threadIdx.x;
    const uint32_t ic = i < n ? i : 0u;         // own loads before staging, so they overlap it
    const uint32_t sn0 = L.stage_n[b];
    const SetIds ids = early_ids(L, b);
    Head hd = list_head(L, c.cap, ic);
    const float4 vi = vel_i[ic];
    const float4 pi = pos[ic];
    const float ki = ws_of(ic);
    list_head_rest(L, sn0, c.cap, ic, hd);
    const uint32_t sn = stage_block<kStageMaxX>(L, b, sn0, ids, [&](uint32_t g) {
        const float4 v = vel_i[g];
        return PV{pos[g], make_float4(v.x, v.y, v.z, ws_of(g))};
    }, [&](uint32_t k, const PV& d) { st.put(k, d); });
    if (i >= n) return;
    if (kvtot) kvtot[i] = ki;
    if (!is_source(L.rs, i)) { vel_o[i] = vi; return; }
    const uint32_t cn = hd.cnt;
    const uint32_t nf = cn & 0xffffu, nb = cn >> 16;
    const uint32_t stride = c.cap;
    float dens = pi.w * c.W0, sg2 = 0.0f, dr = 0.0f;
    float gx = 0.0f, gy = 0.0f, gz = 0.0f, ax = 0.0f, ay = 0.0f, az = 0.0f;
    auto fluid = [&](const float4& pj, const float4& vj, bool valid) {
        const float m = keep(valid, pj.w);
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const PairL kp = pair_listed(c, dist2(dx, dy, dz));
        dens += m * kp.W;
        const float mg = keep(kp.ok, m * kp.g);
        const float px = mg * dx, py = mg * dy, pz = mg * dz;
        sg2 += px * px + py * py + pz * pz;
        gx += px; gy += py; gz += pz;
        dr += (vi.x - vj.x) * px + (vi.y - vj.y) * py + (vi.z - vj.z) * pz;
        if (WS != 2) {
            const float ks = ki + vj.w;
            const float s = keep(fabsf(ks) > kEps, ks);
            ax += s * px; ay += s * py; az += s * pz;
        }
    };
    fluid_nbrs<kStageMaxX>(L, stride, b, i, sn, hd, [&](uint32_t e) { return st.get(e, c.m_uniform); },
               [&](uint32_t j) {
                   const float4 v = vel_i[j];
                   return PV{pos[j], make_float4(v.x, v.y, v.z, ws_of(j))};
               },
               [&](const PV& d, bool valid) { fluid(d.p, d.v, valid); });
    (void)nf;
    float bx = 0.0f, by = 0.0f, bz = 0.0f;
    for_each_nbr32(L.nbrb, stride, i, nb, 0u, hd.b0, hd.b1, [&](uint32_t j) { return load_bnd<SOL>(bpos, L.sol, j); },
        [&](const BN& bj, bool valid) {
        const float4& pj = bj.p;
        const float m = keep(valid, pj.w);
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const PairL kp = pair_listed(c, dist2(dx, dy, dz));
        dens += m * kp.W;
        const float mg = keep(kp.ok, m * kp.g);
        const float px = mg * dx, py = mg * dy, pz = mg * dz;
        sg2 += px * px + py * py + pz * pz;
        gx += px; gy += py; gz += pz;
        dr += (vi.x - bj.v.x) * px + (vi.y - bj.v.y) * py + (vi.z - bj.v.z) * pz;
        bx += px; by += py; bz += pz;
    });
    sg2 += gx * gx + gy * gy + gz * gz;
    const float a = -inv_h / fmaxf(sg2, kEps);
    const float r = (nf + nb < 20u) ? 0.0f : fmaxf(dr, 0.0f);
    rho[i] = dens;
    alpha[i] = a;
    radv[i] = r;
    float4 vo = vi;
    if (WS != 2 && r > 0.0f && is_compute(L.rs, i)) {
        if (fabsf(ki) > kEps) {
            ax += ki * bx; ay += ki * by; az += ki * bz;
            if (SOL) {
                // reactions on the body particles: a second pass, since the
                // gate (a positive source) is known only after the first
                const float mk = -pi.w * ki;
                for_each_nbr32(L.nbrb, stride, i, nb, 0u, [&](uint32_t j) { return load_bnd<SOL>(bpos, L.sol, j); },
                    [&](const BN& bj, bool valid) {
                    const float dx = pi.x - bj.p.x, dy = pi.y - bj.p.y, dz = pi.z - bj.p.z;
                    const PairL kp = grad_listed(c, dist2(dx, dy, dz));
                    const float f = keep(valid && kp.ok, mk * bj.p.w * kp.g);
                    add_reaction<SOL>(L.sol, bj.v, valid, f * dx, f * dy, f * dz);
                });
            }
        }
        vo.x += h * ax; vo.y += h * ay; vo.z += h * az;
    }
    vel_o[i] = vo;
}

// Divergence source from the current velocities: computeDensityChange
// (DFSPH_core_cuda.cu:546-614) in DFSPH_divergence_init_kernel (:618-709, INIT:
// kappaV = 0) and DFSPH_divergence_loop_end_kernel (:732-748) + the FP64 error
// reduction that replaces cub::DeviceReduce::Sum + cudaMemcpy (:774-781).
// Also stores k_i = rho_adv_i * alpha_i for the next Jacobi sweep.
template <bool INIT, bool SOL, bool UM>
__global__ __launch_bounds__(kBlock, UM ? DFSPH_PV_WAVES : 1) void k_div_source(SimConst c, uint32_t n, const float4* __restrict__ pos,
                                                       const float4* __restrict__ bpos, NbrLists L,
                                                       const float4* __restrict__ vel,
                                                       const float* __restrict__ alpha,
                                                       float* __restrict__ radv, float* __restrict__ kk,
                                                       float* __restrict__ kappaV, SolveCtl* ctl,
                                                       double* partial, CtlInit ci)
{
    if (INIT && ci.sc && blockIdx.x == 0 && threadIdx.x == 0) ctl_init(ci);
    __shared__ double lds4[kBlock / 64];
    __shared__ PVStage<UM> st;
    if (!INIT && ctl->done) return;
    const uint32_t b = xcd_block();
    const uint32_t i = b * kBlock + threadIdx.x;
    const uint32_t ic = i < n ? i : 0u;         // own loads before staging, so they overlap it
    const uint32_t sn0 = L.stage_n[b];
    const SetIds ids = early_ids(L, b);
    Head hd = list_head(L, c.cap, ic);
    const float4 pi = pos[ic];
    const float4 vi = vel[ic];
    const float ai = alpha[ic];
    list_head_rest(L, sn0, c.cap, ic, hd);
    const uint32_t sn = stage_block<kStageMaxPV>(L, b, sn0, ids, [&](uint32_t g) { return PV{pos[g], vel[g]}; },
                                    [&](uint32_t k, const PV& d) { st.put(k, d); });
    float r = 0.0f;
    if (i < n && !is_source(L.rs, i)) r = radv[i];      // restricted out: stored value in the error sum
    if (i < n && is_source(L.rs, i)) {
        const uint32_t cn = hd.cnt;
        const uint32_t nf = cn & 0xffffu, nb = cn >> 16;
        // with a uniform mass the fluid sum is taken without it and scaled once
        float dr = 0.0f;
        auto fluid = [&](const float4& pj, const float4& vj, bool valid) {
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const PairL kp = grad_listed(c, dist2(dx, dy, dz));
            const float mg = keep(valid && kp.ok, UM ? kp.g : pj.w * kp.g);
            dr += mg * ((vi.x - vj.x) * dx + (vi.y - vj.y) * dy + (vi.z - vj.z) * dz);
        };
        fluid_nbrs<kStageMaxPV>(L, c.cap, b, i, sn, hd, [&](uint32_t e) { return st.get(e, c.m_uniform); },
                   [&](uint32_t j) { return PV{pos[j], vel[j]}; },
                   [&](const PV& d, bool valid) { fluid(d.p, d.v, valid); });
        if (UM) dr *= c.m_uniform;
        for_each_nbr32(L.nbrb, c.cap, i, nb, 0u, hd.b0, hd.b1,
            [&](uint32_t j) { return load_bnd<SOL>(bpos, L.sol, j); }, [&](const BN& bj, bool valid) {
            const float4& pj = bj.p;
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const PairL kp = grad_listed(c, dist2(dx, dy, dz));
            const float mg = keep(valid && kp.ok, pj.w * kp.g);
            dr += mg * ((vi.x - bj.v.x) * dx + (vi.y - bj.v.y) * dy + (vi.z - bj.v.z) * dz);
        });
        r = (nf + nb < 20u) ? 0.0f : fmaxf(dr, 0.0f);
        radv[i] = r;
        kk[i] = r * ai;
        if (INIT) kappaV[i] = 0.0f;
    }
    if (!INIT) {
        const double bs = block_sum((double)r, lds4);
        store_partial(partial, bs);
    }
}

// End of a solve: the step's total = applied warm start + the solver's
// accumulated increments, in dt-invariant units (scale h for kappaV, h_f^2 for kappa).
__device__ __forceinline__ void finish_total(const DevTime& t, bool pressure, const Totals& f, uint32_t i)
{
    const float s = pressure ? t.h_future * t.h_future : t.h;
    f.tot[i] = (f.tot[i] + f.inc[i]) * s;
}

__global__ void k_finish_totals(const DevTime* t, uint32_t n, int pressure, Totals f)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) finish_total(*t, pressure != 0, f, i);
}

// Jacobi velocity update: divergenceSolveParticle<false> (DFSPH_core_cuda.cu:400-481,
// DIV: kappaV += k_i, step h) and pressureSolveParticle<false> (:867-951, step h_future):
// v_i += step (sum_f [|k_i + k_j| > eps] (k_i + k_j) m_j gradW + [|k_i| > eps] sum_b k_i psi_j gradW)
// The sweep queued before the loop's end is known (fin.tot given) takes the
// step's totals instead of the iteration when the loop has ended.
template <bool DIV, bool SOL, bool UM>
__global__ __launch_bounds__(kBlock) void k_jacobi(SimConst c, const DevTime* t, uint32_t n,
                                                   const float4* __restrict__ pos,
                                                   const float4* __restrict__ bpos, NbrLists L,
                                                   const float* __restrict__ kk, float* __restrict__ kappaV,
                                                   float4* __restrict__ vel, const SolveCtl* ctl, Totals fin)
{
    __shared__ PKStage<UM> st;
    const uint32_t b = xcd_block();
    const uint32_t i = b * kBlock + threadIdx.x;
    if (ctl->done) {
        if (fin.tot && i < n) finish_total(*t, !DIV, fin, i);
        return;
    }
    const uint32_t ic = i < n ? i : 0u;         // own loads before staging, so they overlap it
    const uint32_t sn0 = L.stage_n[b];
    const SetIds ids = early_ids(L, b);
    const float ki = kk[ic];
    const float kv = DIV ? kappaV[ic] : 0.0f;
    const float4 pi = pos[ic];
    float4 v = vel[ic];
    const uint32_t sn = stage_block(L, b, sn0, ids, [&](uint32_t g) { return PK{pos[g], kk[g]}; },
                                    [&](uint32_t k, const PK& d) { st.put(k, d); });
    if (i >= n || !is_compute(L.rs, i)) return;
    if (DIV) kappaV[i] = kv + ki;
    const uint32_t cn = L.cnt[i];
    const uint32_t nf = cn & 0xffffu, nb = cn >> 16;
    // with a uniform mass the fluid sum is taken without it and scaled once
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    auto fluid = [&](const float4& pj, float kj, bool valid) {
        const float ks = ki + kj;
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const PairL kp = grad_listed(c, dist2(dx, dy, dz));
        const float s = keep(valid && kp.ok && fabsf(ks) > kEps, UM ? ks * kp.g : ks * pj.w * kp.g);
        ax += s * dx; ay += s * dy; az += s * dz;
    };
    fluid_nbrs(L, c.cap, b, i, nf, sn, [&](uint32_t e) { return st.get(e, c.m_uniform); },
               [&](uint32_t j) { return PK{pos[j], kk[j]}; },
               [&](const PK& d, bool valid) { fluid(d.p, d.k, valid); });
    if (UM) { ax *= c.m_uniform; ay *= c.m_uniform; az *= c.m_uniform; }
    if (fabsf(ki) > kEps) {
        const float mi = pi.w;
        for_each_nbr32(L.nbrb, c.cap, i, nb, 0u, [&](uint32_t j) { return load_bnd<SOL>(bpos, L.sol, j); },
            [&](const BN& bj, bool valid) {
            const float4& pj = bj.p;
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const PairL kp = grad_listed(c, dist2(dx, dy, dz));
            const float s = keep(valid && kp.ok, ki * pj.w * kp.g);
            ax += s * dx; ay += s * dy; az += s * dz;
            add_reaction<SOL>(L.sol, bj.v, valid, -mi * s * dx, -mi * s * dy, -mi * s * dz);
        });
    }
    const float step = DIV ? t->h : t->h_future;
    v.x += step * ax; v.y += step * ay; v.z += step * az;
    vel[i] = v;
}

// DFSPH_viscosityXSPH_kernel (DFSPH_core_cuda.cu:1423-1510):
// a_i = g - sum_f (1/h) nu (m_j / rho_j) (v_i - v_j) W_ij, fused with the CFL
// block maxima of |v + a h|^2 (DFSPH_CFLVelSquaredNorm_kernel, :3273-3278), which
// k_time_update reduces.
__global__ __launch_bounds__(kBlock, DFSPH_PV_WAVES) void k_xsph(SimConst c, const DevTime* t, uint32_t n,
                                                 const float4* __restrict__ pos, NbrLists L,
                                                 const float4* __restrict__ vel,
                                                 const float* __restrict__ rho, float4* __restrict__ acc,
                                                 DevCtl* ctl, float* partial)
{
    __shared__ float lds4[kBlock / 64];
    __shared__ PVSStage<true> st;                // (x, v, m / rho) of the staged set (the mass is not used)
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->escaped = 0;   // counted afresh by the step's update_pos
    const uint32_t b = xcd_block();
    const uint32_t i = b * kBlock + threadIdx.x;
    const uint32_t ic = i < n ? i : 0u;         // own loads before staging, so they overlap it
    const uint32_t sn0 = L.stage_n[b];
    const SetIds ids = early_ids(L, b);
    Head hd = list_head(L, c.cap, ic);
    const float4 pi = pos[ic];
    const float4 vi = vel[ic];
    list_head_rest(L, sn0, c.cap, ic, hd);
    const uint32_t sn = stage_block<kStageMaxX>(L, b, sn0, ids, [&](uint32_t g) {
        const float4 p = pos[g];
        const float4 v = vel[g];
        return PV{p, make_float4(v.x, v.y, v.z, p.w / rho[g])};
    }, [&](uint32_t k, const PV& d) { st.put(k, d); });
    float m2 = 0.0f;
    if (i < n && !is_compute(L.rs, i)) {
        // restricted out: its stored acceleration still enters the CFL bound
        // (the reference's maximum runs over all particles, DFSPH_core_cuda.cu:3340-3355)
        const float4 a = acc[i];
        const float h = t->h;
        const float wx = vi.x + a.x * h, wy = vi.y + a.y * h, wz = vi.z + a.z * h;
        m2 = wx * wx + wy * wy + wz * wz;
    }
    if (i < n && is_compute(L.rs, i)) {
        const float coef = t->inv_h * c.viscosity;
        float ax = 0.0f, ay = 0.0f, az = 0.0f;
        auto fluid = [&](const float4& pj, const float4& vj, bool valid) {
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const float w = W_listed(c, dist2(dx, dy, dz));
            const float s = keep(valid, coef * vj.w * w);
            ax -= s * (vi.x - vj.x); ay -= s * (vi.y - vj.y); az -= s * (vi.z - vj.z);
        };
        fluid_nbrs<kStageMaxX>(L, c.cap, b, i, sn, hd, [&](uint32_t e) { return st.get(e, 0.0f); },
                   [&](uint32_t j) {
                       const float4 p = pos[j];
                       const float4 v = vel[j];
                       return PV{p, make_float4(v.x, v.y, v.z, p.w / rho[j])};
                   },
                   [&](const PV& d, bool valid) { fluid(d.p, d.v, valid); });
        const float4 a = make_float4(c.gx + ax, c.gy + ay, c.gz + az, 0.0f);
        acc[i] = a;
        const float h = t->h;
        const float wx = vi.x + a.x * h, wy = vi.y + a.y * h, wz = vi.z + a.z * h;
        m2 = wx * wx + wy * wy + wz * wz;
    }
    float m = wave_max(m2);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) lds4[w] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float bm = lds4[0];
        for (int k = 1; k < kBlock / 64; ++k) bm = fmaxf(bm, lds4[k]);
        partial[blockIdx.x] = bm;
    }
}

// DFSPH_update_vel_kernel (DFSPH_core_cuda.cu:3047-3070): v += h a and the
// pressure warm-start rescale kappa = max(kappa h^2 / h_f^2, -0.5).
__global__ void k_update_vel(const DevTime* t, uint32_t n, const float4* acc, float4* vel, float* kappa, Restrict rs)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !is_compute(rs, i)) return;
    const float h = t->h;
    const float4 a = acc[i];
    float4 v = vel[i];
    v.x += h * a.x; v.y += h * a.y; v.z += h * a.z;
    vel[i] = v;
    kappa[i] = fmaxf(kappa[i] * t->ratio2, -0.5f);
}

// Pressure warm start cuda_pressure_compute<true> (DFSPH_core_cuda.cu:965-1000,
// pressureSolveParticle<true> :867-951), optionally fused with the velocity
// update of DFSPH_update_vel_kernel (APPLY_ACC):
// v_i += h a_i;  v_i += h_f (sum_f [|k_i+k_j|>eps] (k_i+k_j) m_j gradW + [|k_i|>eps] sum_b k_i psi_j gradW)
// with k = max(kappa ratio2, -0.5) (WS == 0; ratio2 = 1 when already applied),
// or that value plus the learned correction, bounded by ws_learned (WS == 1).
// kws holds the last solve's kappa increments.  No gate (unlike the divergence
// warm start).  The applied k_i starts the particle's total of the step in
// ktot (when given).
// With a uniform mass the stage is the Jacobi sweep's 16-byte records, 52 KB, which
// fit three blocks per CU where 20-byte ones fit two.  The plain warm start
// without bodies keeps to their 80 registers too (4.19 M particles 203 -> 173 us); with
// bodies or the learned start and the velocity update it takes 81 to 84 and two
// blocks (held to 80 it spills: wave tank of 260k 20 us, 150k learned 16 to 17, both either way).
template <int WS, bool APPLY_ACC, bool SOL, bool UM>
__global__ __launch_bounds__(kBlock) void k_pressure_ws(SimConst c, const DevTime* t, uint32_t n,
                                                        const float4* __restrict__ pos,
                                                        const float4* __restrict__ bpos, NbrLists L,
                                                        const float4* __restrict__ acc,
                                                        float4* __restrict__ vel,
                                                        const float* __restrict__ kws, WsLearned lw, int rescale,
                                                        float* __restrict__ ktot)
{
    __shared__ PKStage<UM> st;
    const float ratio2 = rescale ? t->ratio2 : 1.0f;
    const float ihf2 = t->inv_h_future * t->inv_h_future;
    auto ws_of = [&](uint32_t j) -> float {
        const float ref = fmaxf(kws[j] * ratio2, -0.5f);
        if (WS == 0) return ref;
        return ws_learned(ref, fmaxf(lw.prev[j] * ihf2, -0.5f), lw.dy[j] * lw.scale * ihf2);
    };
    const uint32_t b = xcd_block();
    const uint32_t i = b * kBlock + threadIdx.x;
    const uint32_t ic = i < n ? i : 0u;         // own loads before staging, so they overlap it
    const uint32_t sn0 = L.stage_n[b];
    const SetIds ids = early_ids(L, b);
    const float ki = ws_of(ic);
    const float4 pi = pos[ic];
    float4 v = vel[ic];
    const float4 aown = APPLY_ACC ? acc[ic] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const uint32_t sn = stage_block(L, b, sn0, ids, [&](uint32_t g) { return PK{pos[g], ws_of(g)}; },
                                    [&](uint32_t k, const PK& d) { st.put(k, d); });
    if (i >= n || !is_compute(L.rs, i)) return;
    if (ktot) ktot[i] = ki;
    const uint32_t cn = L.cnt[i];
    const uint32_t nf = cn & 0xffffu, nb = cn >> 16;
    float ax = 0.0f, ay = 0.0f, az = 0.0f;
    auto fluid = [&](const float4& pj, float kj, bool valid) {
        const float ks = ki + kj;
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const PairL kp = grad_listed(c, dist2(dx, dy, dz));
        const float s = keep(valid && kp.ok && fabsf(ks) > kEps, ks * pj.w * kp.g);
        ax += s * dx; ay += s * dy; az += s * dz;
    };
    fluid_nbrs(L, c.cap, b, i, nf, sn, [&](uint32_t e) { return st.get(e, c.m_uniform); },
               [&](uint32_t j) { return PK{pos[j], ws_of(j)}; },
               [&](const PK& d, bool valid) { fluid(d.p, d.k, valid); });
    if (fabsf(ki) > kEps) {
        const float mi = pi.w;
        for_each_nbr32(L.nbrb, c.cap, i, nb, 0u, [&](uint32_t j) { return load_bnd<SOL>(bpos, L.sol, j); },
            [&](const BN& bj, bool valid) {
            const float4& pj = bj.p;
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const PairL kp = grad_listed(c, dist2(dx, dy, dz));
            const float s = keep(valid && kp.ok, ki * pj.w * kp.g);
            ax += s * dx; ay += s * dy; az += s * dz;
            add_reaction<SOL>(L.sol, bj.v, valid, -mi * s * dx, -mi * s * dy, -mi * s * dz);
        });
    }
    if (APPLY_ACC) {
        const float h = t->h;
        const float4 a = aown;
        v.x += h * a.x; v.y += h * a.y; v.z += h * a.z;
    }
    const float hf = t->h_future;
    v.x += hf * ax; v.y += hf * ay; v.z += hf * az;
    vel[i] = v;
}

// Density source computeDensityAdv (DFSPH_core_cuda.cu:1165-1215):
// rho_adv = max(rho + h_f sum m_j (v_i - v_j).gradW - rho0, 0); kappa += rho_adv alpha.
// INIT: DFSPH_pressure_init_kernel (:1217-1262): alpha *= 1/h_f, kappa = 0 first.
// Otherwise DFSPH_pressure_loop_end_kernel (:1264-1284) + FP64 error reduction
// (replaces cub Sum + cudaMemcpy, :1321-1325).
template <bool INIT, bool SOL, bool UM>
__global__ __launch_bounds__(kBlock, UM ? DFSPH_PV_WAVES : 1) void k_density_source(SimConst c, const DevTime* t, uint32_t n,
                                                           const float4* __restrict__ pos,
                                                           const float4* __restrict__ bpos, NbrLists L,
                                                           const float4* __restrict__ vel,
                                                           const float* __restrict__ rho,
                                                           float* __restrict__ alpha, float* __restrict__ radv,
                                                           float* __restrict__ kk, float* __restrict__ kappa,
                                                           SolveCtl* ctl, double* partial, CtlInit ci)
{
    if (INIT && ci.sc && blockIdx.x == 0 && threadIdx.x == 0) ctl_init(ci);
    __shared__ double lds4[kBlock / 64];
    __shared__ PVStage<UM> st;
    if (!INIT && ctl->done) return;
    const uint32_t b = xcd_block();
    const uint32_t i = b * kBlock + threadIdx.x;
    const uint32_t ic = i < n ? i : 0u;         // own loads before staging, so they overlap it
    const uint32_t sn0 = L.stage_n[b];
    const SetIds ids = early_ids(L, b);
    Head hd = list_head(L, c.cap, ic);
    const float4 pi = pos[ic];
    const float4 vi = vel[ic];
    const float a0 = alpha[ic], rho_i = rho[ic];
    const float kap0 = INIT ? 0.0f : kappa[ic];
    list_head_rest(L, sn0, c.cap, ic, hd);
    const uint32_t sn = stage_block<kStageMaxPV>(L, b, sn0, ids, [&](uint32_t g) { return PV{pos[g], vel[g]}; },
                                    [&](uint32_t k, const PV& d) { st.put(k, d); });
    float r = 0.0f;
    if (i < n && !is_source(L.rs, i)) r = radv[i];      // restricted out: stored value in the error sum
    if (i < n && is_source(L.rs, i)) {
        const float hf = t->h_future;
        const uint32_t cn = hd.cnt;
        const uint32_t nf = cn & 0xffffu, nb = cn >> 16;
        // with a uniform mass the fluid sum is taken without it and scaled once
        float dr = 0.0f;
        auto fluid = [&](const float4& pj, const float4& vj, bool valid) {
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const PairL kp = grad_listed(c, dist2(dx, dy, dz));
            const float mg = keep(valid && kp.ok, UM ? kp.g : pj.w * kp.g);
            dr += mg * ((vi.x - vj.x) * dx + (vi.y - vj.y) * dy + (vi.z - vj.z) * dz);
        };
        fluid_nbrs<kStageMaxPV>(L, c.cap, b, i, sn, hd, [&](uint32_t e) { return st.get(e, c.m_uniform); },
                   [&](uint32_t j) { return PV{pos[j], vel[j]}; },
                   [&](const PV& d, bool valid) { fluid(d.p, d.v, valid); });
        if (UM) dr *= c.m_uniform;
        (void)nf;
        for_each_nbr32(L.nbrb, c.cap, i, nb, 0u, hd.b0, hd.b1,
            [&](uint32_t j) { return load_bnd<SOL>(bpos, L.sol, j); }, [&](const BN& bj, bool valid) {
            const float4& pj = bj.p;
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const PairL kp = grad_listed(c, dist2(dx, dy, dz));
            const float mg = keep(valid && kp.ok, pj.w * kp.g);
            dr += mg * ((vi.x - bj.v.x) * dx + (vi.y - bj.v.y) * dy + (vi.z - bj.v.z) * dz);
        });
        float a = a0;
        if (INIT) { a *= t->inv_h_future; alpha[i] = a; }
        r = fmaxf(rho_i + hf * dr - c.density0, 0.0f);
        radv[i] = r;
        const float ka = r * a;
        kk[i] = ka;
        kappa[i] = INIT ? ka : kap0 + ka;
    }
    if (!INIT) {
        const double bs = block_sum((double)r, lds4);
        store_partial(partial, bs);
    }
}

// DFSPH_update_pos_kernel (DFSPH_core_cuda.cu:3127-3214): x += h v, fused with the
// escape count of tag_particles_outside_bounding_box_kernel
// (SPH_other_systems_cuda.cu:1244-1281): outside if any coordinate leaves the box.
__global__ void k_update_pos(const DevTime* t, uint32_t n, const float4* vel, float4* pos,
                             float bx0, float by0, float bz0, float bx1, float by1, float bz1, DevCtl* ctl,
                             Restrict rs)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t out = 0;
    if (i < n) {
        const float h = t->h;
        const float4 v = vel[i];
        float4 x = pos[i];
        if (is_compute(rs, i)) {
            x.x += h * v.x; x.y += h * v.y; x.z += h * v.z;
            pos[i] = x;
        }
        out = (x.x > bx1 || x.y > by1 || x.z > bz1 || x.x < bx0 || x.y < by0 || x.z < bz0) ? 1u : 0u;
    }
    const uint32_t s = wave_sum_u(out);
    if ((threadIdx.x & 63) == 0 && s) atomicAdd(&ctl->escaped, s);
}

// keep flags for the compaction (tag_particles_outside_bounding_box_kernel)
__global__ void k_keep_inside(uint32_t n, const float4* pos, float bx0, float by0, float bz0,
                              float bx1, float by1, float bz1, uint32_t* keep)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    if (i == n) { keep[n] = 0; return; }
    const float4 x = pos[i];
    const bool out = x.x > bx1 || x.y > by1 || x.z > bz1 || x.x < bx0 || x.y < by0 || x.z < bz0;
    keep[i] = out ? 0u : 1u;
}

__global__ void k_keep_from_u8(uint32_t n, const uint8_t* k8, uint32_t* keep)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > n) return;
    keep[i] = (i < n && k8[i]) ? 1u : 0u;
}

// Stable compaction: the kept particles move to their exclusive-scan rank
// (replaces the radix sort by tag + cuda_sortData of remove_tagged_particles,
// SPH_other_systems_cuda.cu:1606-1641).
__global__ void k_compact(uint32_t n, const uint32_t* keep, const uint32_t* rank, FluidPtrs in, FluidPtrs out)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || !keep[i]) return;
    copy_fluid(in, i, out, rank[i]);
}

// Features of the learned warm start, one neighbor sweep over the current state
// (before the divergence warm start):
//  0 rho / rho0 - 1            1 divergence source h / rho0 (unclamped)
//  2 (n_fluid + n_boundary) / 40   3 |v| h / (2r)
//  4 last density increments kappa h_f^2 / d^2   5 last divergence increments kappaV h / d
//  6 boundary fraction n_b / n     7-9 mean neighbor offset / h_k
// 10 mean neighbor distance / h_k 11 fluid share of the density
template <bool SOL, bool UM>
__global__ __launch_bounds__(kBlock, UM ? DFSPH_PV_WAVES : 1) void k_features(SimConst c, const DevTime* t, uint32_t n,
                                                     const float4* __restrict__ pos,
                                                     const float4* __restrict__ bpos, NbrLists L,
                                                     const float4* __restrict__ vel,
                                                     const float* __restrict__ kap,
                                                     const float* __restrict__ kapv,
                                                     const float* __restrict__ ktot,
                                                     const float* __restrict__ kvtot, float diameter,
                                                     float* __restrict__ feat, float* __restrict__ prev_p,
                                                     float* __restrict__ prev_v)
{
    __shared__ PVStage<UM> st;
    const uint32_t b = xcd_block();
    const uint32_t i = b * kBlock + threadIdx.x;
    const uint32_t ic = i < n ? i : 0u;         // own loads before staging, so they overlap it
    const uint32_t sn0 = L.stage_n[b];
    const SetIds ids = early_ids(L, b);
    Head hd = list_head(L, c.cap, ic);
    const float4 pi = pos[ic];
    const float4 vi = vel[ic];
    list_head_rest(L, sn0, c.cap, ic, hd);
    const uint32_t sn = stage_block<kStageMaxPV>(L, b, sn0, ids, [&](uint32_t g) { return PV{pos[g], vel[g]}; },
                                    [&](uint32_t k, const PV& d) { st.put(k, d); });
    if (i >= n) return;
    const uint32_t cn = hd.cnt;
    const uint32_t nf = cn & 0xffffu, nb = cn >> 16;
    float dens = pi.w * c.W0, dfl = 0.0f, dr = 0.0f;
    float ox = 0.0f, oy = 0.0f, oz = 0.0f, od = 0.0f;
    auto fluid = [&](const float4& pj, const float4& vj, bool valid) {
        const float m = keep(valid, 1.0f);
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const float r2 = dist2(dx, dy, dz);
        const PairL kp = pair_listed(c, r2);
        const float mj = m * pj.w;
        dfl += mj * kp.W;
        dr += keep(kp.ok, mj * kp.g) * ((vi.x - vj.x) * dx + (vi.y - vj.y) * dy + (vi.z - vj.z) * dz);
        ox -= m * dx; oy -= m * dy; oz -= m * dz;
        od += m * __builtin_sqrtf(r2);
    };
    fluid_nbrs<kStageMaxPV>(L, c.cap, b, i, sn, hd, [&](uint32_t e) { return st.get(e, c.m_uniform); },
               [&](uint32_t j) { return PV{pos[j], vel[j]}; },
               [&](const PV& d, bool valid) { fluid(d.p, d.v, valid); });
    float dbd = 0.0f;
    for_each_nbr32(L.nbrb, c.cap, i, nb, 0u, hd.b0, hd.b1, [&](uint32_t j) { return load_bnd<SOL>(bpos, L.sol, j); },
        [&](const BN& bj, bool valid) {
        const float4& pj = bj.p;
        const float m = keep(valid, 1.0f);
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const float r2 = dist2(dx, dy, dz);
        const PairL kp = pair_listed(c, r2);
        const float mj = m * pj.w;
        dbd += mj * kp.W;
        dr += keep(kp.ok, mj * kp.g) * ((vi.x - bj.v.x) * dx + (vi.y - bj.v.y) * dy + (vi.z - bj.v.z) * dz);
        ox -= m * dx; oy -= m * dy; oz -= m * dz;
        od += m * __builtin_sqrtf(r2);
    });
    dens += dfl + dbd;
    const float nn = (float)(nf + nb);
    const float inv_n = nn > 0.0f ? 1.0f / nn : 0.0f;
    const float s = c.inv_hk * inv_n;
    float* f = feat + (size_t)i * 12;
    f[0] = dens / c.density0 - 1.0f;
    f[1] = dr * t->h / c.density0;
    f[2] = nn * (1.0f / 40.0f);
    f[3] = __builtin_sqrtf(vi.x * vi.x + vi.y * vi.y + vi.z * vi.z) * t->h / diameter;
    const float inv_d = 1.0f / diameter;
    f[kFeatKappaP] = kap[i] * (t->h * t->h) * (inv_d * inv_d);
    f[kFeatKappaV] = kapv[i] * t->h_past * inv_d;
    f[6] = (float)nb * inv_n;
    f[7] = ox * s;
    f[8] = oy * s;
    f[9] = oz * s;
    f[10] = od * s;
    f[11] = dfl / dens;
    prev_p[i] = ktot[i];
    prev_v[i] = kvtot[i];
}

// training set, after a step's solves with the reference warm start: append
// the step's features and the solves' increments in dt-invariant units
// (kappaV h, kappa h_f^2), what the reference warm start left to the Jacobi
// iterations: the correction the network learns
__global__ void k_harvest(const DevTime* t, uint32_t n, uint32_t stride, uint32_t offset, uint32_t cap,
                          const float* feat, const float* kapv, const float* kap, float inv_d, float* ds_x,
                          float* ds_t)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t i = k * stride;
    if (i >= n || offset + k >= cap) return;
    const size_t o = offset + k;
    const float* f = feat + (size_t)i * 12;
    for (int a = 0; a < 12; ++a) ds_x[o * 12 + a] = f[a];
    ds_t[o * 2 + 0] = kapv[i] * t->h * inv_d;
    ds_t[o * 2 + 1] = kap[i] * (t->h_future * t->h_future) * (inv_d * inv_d);
}

// ------------------------------------------------------------------------
// host launch wrappers
// ------------------------------------------------------------------------
static inline uint32_t nblk(uint32_t n) { return (n + kBlock - 1) / kBlock; }
static inline uint32_t nblk_xcd(uint32_t n)
{
    const uint32_t b = nblk(n);
    return ((b + kNumXcd - 1) / kNumXcd) * kNumXcd;
}

uint32_t grid_blocks_xcd(uint32_t n) { return nblk_xcd(n ? n : 1); }

// Blocks that share a set in the search of n particles: as long as the blocks
// leave CUs idle, the candidate tests and list writing of a block's wavefronts
// (most of its time, at the rate of its CU's vector units) go to several, each
// with its own copy of the set.  16k particles: 39 us with one, 37 with eight
// (a step 333 -> 317 us); 1600 particles: a step 289 -> 284 us.
uint32_t search_split(uint32_t n)
{
    uint32_t split = 1;
    while (split < kBlock / 64u && nblk(n) * split * 2u <= kNumCu) split *= 2u;
    return split;
}

// What the sweeps over n particles read past the caches (non-temporal loads).
// A pass reads some 128 bytes a particle, the 16-bit lists among them, and the passes
// of a step read the same again: up to the 256 MB of the memory-side cache
// it stays there.  Beyond, the lists (read once a pass) drive out the records
// that the blocks' sets are gathered from; the rest, some 85 bytes, fits longer, and
// then the sets' ids go the same way.  Both sides, divergence (4 iterations) plus density
// solve (3), us, at 29 neighbors and walls at spacing 2r (r):
//   n, M       1.46        1.83        2.12        2.81        3.20        3.63        4.19        5.73
//   cached     924 (1071) 1185 (1382) 1392 (1636) 1881 (2153) 2146 (2406) 2433 (2772) 2804 (3163) 3747 (4200)
//   lists      985 (1128) 1195 (1358) 1338 (1508) 1690 (1928) 1956 (2218) 2227 (2560) 2624 (2982) 3606 (4098)
//   and ids   1006 (1141) 1223 (1376) 1368 (1535) 1723 (1917) 1939 (2157) 2150 (2463) 2483 (2859) 3496 (4025)
uint32_t list_stream(uint32_t n)
{
    constexpr uint32_t kPassBytes = 128u, kRestBytes = 85u, kCacheBytes = 1u << 28;
    if (n < kCacheBytes / kPassBytes) return 0u;
    return n < kCacheBytes / kRestBytes ? kStreamLists : kStreamLists | kStreamIds;
}

static thread_local hipEvent_t tl_ev_start = nullptr, tl_ev_stop = nullptr;

void arm_sweep_events(hipEvent_t start, hipEvent_t stop)
{
    tl_ev_start = start;
    tl_ev_stop = stop;
}
bool sweep_events_armed() { return tl_ev_start != nullptr; }
void disarm_sweep_events() { tl_ev_start = tl_ev_stop = nullptr; }

// A sweep launch of g blocks of kBlock threads; it takes the armed timing
// events, if any, into its dispatch.
template <class... P, class... A>
static void sweep_launch(void (*k)(P...), uint32_t g, hipStream_t s, A... a)
{
    if (tl_ev_start) {
        hipExtLaunchKernelGGL(k, dim3(g), dim3(kBlock), 0u, s, tl_ev_start, tl_ev_stop, 0u, a...);
        disarm_sweep_events();
    } else {
        k<<<g, kBlock, 0, s>>>(a...);
    }
}

void launch_fill_u32(hipStream_t s, uint32_t* p, uint32_t v, uint32_t n)
{
    if (n) k_fill_u32<<<nblk(n), kBlock, 0, s>>>(p, v, n);
}

void launch_fill_f32(hipStream_t s, float* p, float v, uint32_t n)
{
    if (n) k_fill_f32<<<nblk(n), kBlock, 0, s>>>(p, v, n);
}

size_t scan_temp_words(uint32_t n)
{
    size_t words = 0;
    uint32_t m = n;
    while (m > 1) {
        const uint32_t tiles = (m + kScanTile - 1) / kScanTile;
        words += 2 * (size_t)tiles + 2;
        m = tiles;
    }
    return words + 4;
}

void launch_exclusive_scan(hipStream_t s, uint32_t* in, uint32_t* out, uint32_t n, uint32_t* tmp, bool clear_in)
{
    if (n == 0) return;
    const uint32_t tiles = (n + kScanTile - 1) / kScanTile;
    uint32_t* sums = tmp;
    uint32_t* offs = tmp + tiles + 1;
    k_scan_tiles<<<tiles, kBlock, 0, s>>>(in, out, n, sums, clear_in ? 1 : 0);
    if (tiles > 1 && tiles <= kScanDirect) {
        k_scan_add_direct<<<tiles, kBlock, 0, s>>>(out, n, sums);
    } else if (tiles > 1) {
        launch_exclusive_scan(s, sums, offs, tiles, tmp + 2 * (size_t)tiles + 2, false);
        k_scan_add<<<tiles, kBlock, 0, s>>>(out, n, offs);
    }
}

void launch_nbr_ctl_init(hipStream_t s, DevCtl* c) { k_nbr_ctl_init<<<1, 64, 0, s>>>(c); }

void launch_publish_count(hipStream_t s, const uint32_t* count, HostRecord* rec, uint32_t seq)
{
    k_publish_count<<<1, 64, 0, s>>>(count, rec, seq);
}

void launch_time_reset(hipStream_t s, DevTime* t, double h) { k_time_reset<<<1, 64, 0, s>>>(t, h); }

void launch_time_update(hipStream_t s, DevTime* t, double hf, DevCtl* ctl, const float* partial, uint32_t n, int mode,
                        double cfl_factor, double diameter, double dt_min, double dt_max, double seed)
{
    k_time_update<<<1, kBlock, 0, s>>>(t, hf, ctl, partial, nblk_xcd(n ? n : 1), mode, cfl_factor, diameter, dt_min,
                                       dt_max, seed);
}

void launch_time_step_end(hipStream_t s, DevTime* t, const Publish& pub) { k_time_step_end<<<1, 64, 0, s>>>(t, pub); }

void launch_time_set(hipStream_t s, DevTime* t, double h, double hp, double time)
{
    k_time_set<<<1, 64, 0, s>>>(t, h, hp, time);
}

void launch_cell_hist(hipStream_t s, const SimConst& c, const float4* pos, uint32_t n, uint32_t* key,
                      uint32_t* slot, uint32_t* hist)
{
    if (n) k_cell_hist<<<nblk(n), kBlock, 0, s>>>(c, pos, n, key, slot, hist);
}

void launch_scatter_perm(hipStream_t s, const uint32_t* key, const uint32_t* slot, const uint32_t* cstart,
                         uint32_t n, uint32_t* perm)
{
    if (n) k_scatter_perm<<<nblk(n), kBlock, 0, s>>>(key, slot, cstart, n, perm);
}

void launch_order_perm(hipStream_t s, uint32_t n, const uint32_t* key, const uint32_t* cstart, const uint32_t* perm,
                       uint32_t* out)
{
    if (n) k_order_perm<<<nblk(n), kBlock, 0, s>>>(n, CellOrder{key, cstart, perm}, out);
}

void launch_gather_fluid(hipStream_t s, uint32_t n, const uint32_t* key, const uint32_t* cstart, const uint32_t* perm,
                         const FluidPtrs& in, const FluidPtrs& out)
{
    if (n) k_gather_fluid<<<nblk(n), kBlock, 0, s>>>(n, CellOrder{key, cstart, perm}, in, out);
}

void launch_gather_boundary(hipStream_t s, uint32_t n, const uint32_t* key, const uint32_t* cstart,
                            const uint32_t* perm, const float4* in, float4* out, const float4* vin, float4* vout)
{
    if (n) k_gather_boundary<<<nblk(n), kBlock, 0, s>>>(n, CellOrder{key, cstart, perm}, in, out, vin, vout);
}

void launch_neighbors(hipStream_t s, const SimConst& c, bool indirect, const float4* pos, const uint32_t* cs_f,
                      const uint32_t* perm, const float4* bpos, const uint32_t* cs_b, uint32_t n, uint16_t* nbr16,
                      uint32_t* nbrf, uint32_t* nbrb, uint32_t* cnt, uint32_t* stage_n, uint32_t* stg,
                      const Restrict& rs, uint4* part, DevCtl* ctl)
{
    if (!n) return;
    const uint32_t split = search_split(n), g = nblk_xcd(n) * split;
    if (indirect)
        k_neighbors<true><<<g, kBlock, 0, s>>>(c, pos, cs_f, perm, bpos, cs_b, n, nbr16, nbrf, nbrb, cnt, stage_n, stg,
                                               rs, part, split);
    else
        k_neighbors<false><<<g, kBlock, 0, s>>>(c, pos, cs_f, perm, bpos, cs_b, n, nbr16, nbrf, nbrb, cnt, stage_n, stg,
                                                rs, part, split);
    k_nbr_finalize<<<1, kBlock, 0, s>>>(part, g, ctl);
}

void launch_expand_lists(hipStream_t s, uint32_t n, uint32_t cap, const NbrLists& L, uint32_t* out)
{
    if (n) k_expand_lists<<<nblk(n), kBlock, 0, s>>>(n, cap, L, out);
}

void launch_boundary_psi(hipStream_t s, const SimConst& c, const float4* bpos, const uint32_t* cs_b,
                         uint32_t nb, float* psi)
{
    if (nb) k_boundary_psi<<<nblk(nb), kBlock, 0, s>>>(c, bpos, cs_b, nb, psi);
}

void launch_set_w(hipStream_t s, float4* p, const float* w, uint32_t n)
{
    if (n) k_set_w<<<nblk(n), kBlock, 0, s>>>(p, w, n);
}

void launch_div_ws_init(hipStream_t s, int ws, const SimConst& c, const DevTime* t, uint32_t n,
                        const float4* pos, const float4* bpos, const NbrLists& L,
                        const float4* vel_i, float4* vel_o, const float* kws, const WsLearned& lw,
                        float* rho, float* alpha, float* radv, float* kvtot)
{
    if (!n) return;
    const uint32_t g = nblk_xcd(n);
    const bool sol = L.sol.bvel != nullptr;
    const bool um = c.m_uniform > 0.0f;
#define DWU(W, S, U) sweep_launch(k_div_ws_init<W, S, U>, g, s, c, t, n, pos, bpos, L, vel_i, vel_o, kws, lw, rho, alpha, radv, kvtot)
#define DWS(W, S) do { if (um) DWU(W, S, true); else DWU(W, S, false); } while (0)
    if (ws == 0) { if (sol) DWS(0, true); else DWS(0, false); }
    else if (ws == 1) { if (sol) DWS(1, true); else DWS(1, false); }
    else { if (sol) DWS(2, true); else DWS(2, false); }
#undef DWS
#undef DWU
}

void launch_div_source(hipStream_t s, bool init, const SimConst& c, uint32_t n, const float4* pos,
                       const float4* bpos, const NbrLists& L, const float4* vel,
                       const float* alpha, float* radv, float* kk, float* kappaV, SolveCtl* ctl, double* partial,
                       const CtlInit& ci)
{
    const uint32_t g = nblk_xcd(n ? n : 1);
    const bool sol = L.sol.bvel != nullptr;
    const bool um = c.m_uniform > 0.0f;
#define DS(I, S, U, CI) sweep_launch(k_div_source<I, S, U>, g, s, c, n, pos, bpos, L, vel, alpha, radv, kk, kappaV, ctl, partial, CI)
#define DSU(I, S, CI) do { if (um) DS(I, S, true, CI); else DS(I, S, false, CI); } while (0)
    if (init) { if (sol) DSU(true, true, ci); else DSU(true, false, ci); }
    else { if (sol) DSU(false, true, CtlInit{}); else DSU(false, false, CtlInit{}); }
#undef DSU
#undef DS
}

void launch_solve_finalize(hipStream_t s, uint32_t n, SolveCtl* ctl, const double* partial, uint32_t it,
                           const Publish& pub)
{
    k_solve_finalize<<<1, kBlock, 0, s>>>(ctl, partial, nblk_xcd(n ? n : 1), it, pub);
}

void launch_jacobi(hipStream_t s, bool div, const SimConst& c, const DevTime* t, uint32_t n, const float4* pos,
                   const float4* bpos, const NbrLists& L, const float* kk, float* kappaV,
                   float4* vel, const SolveCtl* ctl, const Totals& fin)
{
    if (!n) return;
    const uint32_t g = nblk_xcd(n);
    const bool sol = L.sol.bvel != nullptr;
    const bool um = c.m_uniform > 0.0f;
#define JA(D, S, U) sweep_launch(k_jacobi<D, S, U>, g, s, c, t, n, pos, bpos, L, kk, kappaV, vel, ctl, fin)
#define JAU(D, S) do { if (um) JA(D, S, true); else JA(D, S, false); } while (0)
    if (div) { if (sol) JAU(true, true); else JAU(true, false); }
    else { if (sol) JAU(false, true); else JAU(false, false); }
#undef JAU
#undef JA
}

void launch_xsph(hipStream_t s, const SimConst& c, const DevTime* t, uint32_t n, const float4* pos,
                 const NbrLists& L, const float4* vel, const float* rho, float4* acc,
                 DevCtl* ctl, float* partial)
{
    const uint32_t g = nblk_xcd(n ? n : 1);
    sweep_launch(k_xsph, g, s, c, t, n, pos, L, vel, rho, acc, ctl, partial);
}

void launch_update_vel(hipStream_t s, const DevTime* t, uint32_t n, const float4* acc, float4* vel, float* kappa,
                       const Restrict& rs)
{
    if (n) k_update_vel<<<nblk(n), kBlock, 0, s>>>(t, n, acc, vel, kappa, rs);
}

void launch_pressure_ws(hipStream_t s, int ws, bool apply_acc, const SimConst& c, const DevTime* t, uint32_t n,
                        const float4* pos, const float4* bpos, const NbrLists& L,
                        const float4* acc, float4* vel, const float* kws, const WsLearned& lw, int rescale,
                        float* ktot)
{
    if (!n) return;
    const uint32_t g = nblk_xcd(n);
    const bool sol = L.sol.bvel != nullptr;
    const bool um = c.m_uniform > 0.0f;
#define PWU(W, A, S, U) sweep_launch(k_pressure_ws<W, A, S, U>, g, s, c, t, n, pos, bpos, L, acc, vel, kws, lw, rescale, ktot)
#define PW(W, A, S) do { if (um) PWU(W, A, S, true); else PWU(W, A, S, false); } while (0)
    if (ws == 1) {
        if (apply_acc) { if (sol) PW(1, true, true); else PW(1, true, false); }
        else { if (sol) PW(1, false, true); else PW(1, false, false); }
    } else {
        if (apply_acc) { if (sol) PW(0, true, true); else PW(0, true, false); }
        else { if (sol) PW(0, false, true); else PW(0, false, false); }
    }
#undef PW
#undef PWU
}

void launch_density_source(hipStream_t s, bool init, const SimConst& c, const DevTime* t, uint32_t n,
                           const float4* pos, const float4* bpos, const NbrLists& L,
                           const float4* vel, const float* rho, float* alpha, float* radv, float* kk,
                           float* kappa, SolveCtl* ctl, double* partial, const CtlInit& ci)
{
    const uint32_t g = nblk_xcd(n ? n : 1);
    const bool sol = L.sol.bvel != nullptr;
    const bool um = c.m_uniform > 0.0f;
#define DN(I, S, U, CI) sweep_launch(k_density_source<I, S, U>, g, s, c, t, n, pos, bpos, L, vel, rho, alpha, radv, kk, kappa, ctl, partial, CI)
#define DNU(I, S, CI) do { if (um) DN(I, S, true, CI); else DN(I, S, false, CI); } while (0)
    if (init) { if (sol) DNU(true, true, ci); else DNU(true, false, ci); }
    else { if (sol) DNU(false, true, CtlInit{}); else DNU(false, false, CtlInit{}); }
#undef DNU
#undef DN
}

void launch_update_pos(hipStream_t s, const DevTime* t, uint32_t n, const float4* vel, float4* pos,
                       const float* bmin, const float* bmax, DevCtl* ctl, const Restrict& rs)
{
    if (n)
        sweep_launch(k_update_pos, nblk(n), s, t, n, vel, pos, bmin[0], bmin[1], bmin[2], bmax[0], bmax[1], bmax[2], ctl,
                     rs);
}

void launch_keep_inside(hipStream_t s, uint32_t n, const float4* pos, const float* bmin, const float* bmax,
                        uint32_t* keep)
{
    k_keep_inside<<<nblk(n + 1), kBlock, 0, s>>>(n, pos, bmin[0], bmin[1], bmin[2], bmax[0], bmax[1], bmax[2], keep);
}

void launch_keep_from_u8(hipStream_t s, uint32_t n, const uint8_t* k8, uint32_t* keep)
{
    k_keep_from_u8<<<nblk(n + 1), kBlock, 0, s>>>(n, k8, keep);
}

void launch_compact(hipStream_t s, uint32_t n, const uint32_t* keep, const uint32_t* rank, const FluidPtrs& in,
                    const FluidPtrs& out)
{
    if (n) k_compact<<<nblk(n), kBlock, 0, s>>>(n, keep, rank, in, out);
}

void launch_finish_totals(hipStream_t s, const DevTime* t, uint32_t n, int pressure, const Totals& f)
{
    if (n) k_finish_totals<<<nblk(n), kBlock, 0, s>>>(t, n, pressure, f);
}

void launch_features(hipStream_t s, const SimConst& c, const DevTime* t, uint32_t n, const float4* pos,
                     const float4* bpos, const NbrLists& L, const float4* vel, const float* kap,
                     const float* kapv, const float* ktot, const float* kvtot, float diameter, float* feat,
                     float* prev_p, float* prev_v)
{
    if (!n) return;
    const bool um = c.m_uniform > 0.0f;
#define KF(S, U) sweep_launch(k_features<S, U>, nblk_xcd(n), s, c, t, n, pos, bpos, L, vel, kap, kapv, ktot, kvtot, \
                                  diameter, feat, prev_p, prev_v)
    if (L.sol.bvel) { if (um) KF(true, true); else KF(true, false); }
    else { if (um) KF(false, true); else KF(false, false); }
#undef KF
}

void launch_harvest(hipStream_t s, const DevTime* t, uint32_t n, uint32_t stride, uint32_t offset, uint32_t cap,
                    const float* feat, const float* kapv, const float* kap, float diameter, float* ds_x,
                    float* ds_t)
{
    const uint32_t m = (n + stride - 1) / stride;
    if (m) k_harvest<<<nblk(m), kBlock, 0, s>>>(t, n, stride, offset, cap, feat, kapv, kap, 1.0f / diameter, ds_x,
                                                ds_t);
}

}  // namespace dfsph
