// gg_grid_bands.hpp -- region gridding with the grid cells in LDS, one wave
// per band of eight rows.
//
// A region (kRegionW x kRegionH cells) is cut into column blocks of kBlockW
// cells and bands of eight rows; a wave owns one (block, band) of a work
// item, 8 x kBlockW cells, in 9 KiB of LDS of its own.  Nothing is shared
// between waves: no barriers, no atomics, and a cell's additions happen in
// visit order.  For each visit whose footprint meets the wave's cells the
// wave walks the footprint in units of 8 rows x 8 lanes: one 16-byte load
// per lane brings the unit's taps straight from the kernel table (two
// complex FP32 taps, or one FP64 tap), the same lanes read their cells from
// LDS, do the multiplies and write them back.
//
// Why this shape.  Where a table serves only a few visits of a region (small
// supports, many w-planes, few visibilities) staging it in LDS does not pay,
// and a strip kernel that keeps the cells in registers spends its time on
// per-visit set-up: it walks the footprint in slots fixed to the grid, 8
// bytes a lane, each with its own address, test and branch.  With the cells
// in LDS the units follow the footprint, so every address but the first is
// an immediate, and the row's last unit needs no mask: table rows are padded
// with zeros to whole units, and LDS rows carry a unit of padding that
// absorbs what runs past the block.  A visit issues exactly the loads it
// needs (one straight-line block per number of units): loads issued for absent
// units and masked off cost as much as real ones (+30% on the whole kernel).
// What binds it, by its counters: large stacks (714 planes) stream their tables
// from beyond L2, at 4.7 TB/s in FP32 (2.15M visibilities, 3.0 ms) and 6.8 TB/s
// in FP64 (215k, 0.86 ms), where a copy moves 4.7; the address unit is busy 56
// and 70% of the time, the vector pipe 49 and 22%, LDS 31 and 21%.  Compensated
// (1M, 128 planes, 1.45 ms) 67, 58 and 46%, and waves wait for issue slots.
// Prefetching the next visit's taps into a second set of registers changed
// nothing, nor did wider (192, 256) or narrower (64, 96) blocks gain; two or
// four waves per workgroup cost 5-20%.
#pragma once

#include "gg_kernels.hpp"

namespace gg {

// TAP: precision of the table's taps and amplitudes; CELL: precision the
// cells accumulate in.
template <typename TAP, typename CELL>
struct BandCfg
{
    static constexpr int kLaneCells = sizeof(TAP) == 4 && sizeof(CELL) == 4 ? 2 : 1;
    static constexpr int kUnitW = 8 * kLaneCells;           // cells of a unit's row
    static constexpr int kBlockW = 64 * kLaneCells;         // columns a wave owns
    static constexpr int kBlocks = 2;                       // column blocks of a region
    static constexpr int kRows = 8;                         // rows a wave owns
    static constexpr int kRegionW = kBlocks * kBlockW;
    static constexpr int kRegionH = 128;
    static constexpr int kBands = kRegionH / kRows;
    static constexpr int kWork = kBlocks * kBands;          // waves' shares of an item
    static constexpr int kTapBytes = 2 * (int)sizeof(TAP);
    static constexpr int kLaneBytes = kTapBytes * kLaneCells;
    static constexpr int kUnitBytes = 8 * kLaneBytes;
    static constexpr int kStride = kBlockW / kLaneCells + 8; // 16-byte words per LDS row
    static constexpr int kMaxUnits = kBlockW / kUnitW + 1;  // units of one row in a block
    static_assert(kRegionW * kRegionH % kMergeCells<float2> == 0, "merge blocks tile a region");
    static_assert(kWork == 32, "shares of an item, whatever the precision");
};

// Visits of a sorted list as the kernel reads them (k_gather_bands):
//   x  byte offset of the tap under the region's row 0 and the footprint's
//      first unit (the lanes of the wave and its rows are added per visit)
//   y  bytes from a region row's taps to the next row's (negative: the
//      table's rows run backwards)
//   z  first footprint row in the region (low 16 bits) and first column of
//      the footprint's first unit (high 16 bits), signed
//   w  table width | kBandMirror | kBandConj
constexpr int kBandMirror = 1 << 16;        // table columns run backwards
constexpr int kBandConj = 1 << 17;          // Im(kernel) negated

// A work item as the kernel reads it, one 32-byte scalar load.
constexpr unsigned kNoSlot = 0xffffffffu;
template <typename T>
struct BandItem
{
    unsigned v0, nv;                 // its visits in the sorted list
    unsigned slot;                   // partial-region slot; kNoSlot: added to the grid
    int x0, y0;                      // the region's first cell
    int grid_size;
    typename V2<T>::t* grid;
};
static_assert(sizeof(BandItem<float>) == 32 && sizeof(BandItem<double>) == 32, "one scalar load");

template <typename TAP, typename CELL>
__global__ __launch_bounds__(64)
void k_grid_bands(const GridArgs<TAP> A)
{
    using C = BandCfg<TAP, CELL>;
    typedef typename V2<TAP>::t T2;
    typedef typename V2<CELL>::t C2;
    constexpr int LC = C::kLaneCells;
    struct __align__(16) Word { CELL v[16 / sizeof(CELL)]; };
    struct Tap { TAP v[2 * LC]; };
    // a unit of padding before the first row; each row's own padding follows
    // it and precedes the next
    __shared__ Word cells[8 + C::kRows * C::kStride];
    const unsigned num_items = ld_const(A.d_num_items, 0);
    const int lane = lane_id();
    const int lr = lane >> 3, lc = lane & 7;
    const int lane_word = lr * C::kStride + lc;
    const int lane_fwd = lc * C::kLaneBytes;
    const __amdgpu_buffer_rsrc_t rs_tab = table_rsrc(A.tables, A.table_bytes);

    // Workgroup b runs on XCD b mod 8.  Each XCD takes whole items, all their
    // shares (band, block) one after the other, so that the shares of one
    // item run side by side on one L2; items go to the XCDs in groups of
    // item_group, as in the strip kernel.  One share per workgroup, balanced
    // by the dispatcher (a persistent grid that took shares from per-XCD
    // counters was 5-120% slower); a launch that only knows a bound of the
    // number of items has fewer workgroups, which stride over the shares.
    const unsigned x = blockIdx.x & 7u, g = A.item_group;
    const unsigned per_xcd = (num_items + 8u * g - 1) / (8u * g) * g;   // item positions per XCD
    for (unsigned n = blockIdx.x >> 3; n / C::kWork < per_xcd; n += gridDim.x >> 3)
    {
        const unsigned pos = n / C::kWork, share = n % C::kWork;
        const unsigned at = (pos / g * 8u + x) * g + pos % g;
        if (at >= num_items) continue;
        const int band = (int)(share / C::kBlocks), block = (int)(share % C::kBlocks);
        const BandItem<TAP> I = ld_const(A.band_items, at);
        const unsigned v0 = I.v0, nv = I.nv;
        const int G = I.grid_size;
        const int col0 = block * C::kBlockW, row0 = band * C::kRows;    // in the region
        {
            Word z;
            for (auto& q : z.v) q = (CELL)0;
            for (int i = lane; i < C::kRows * C::kStride; i += 64) cells[8 + i] = z;
        }
        wave_lds_fence();

        // (resources based at the item's records: reads past its last visit
        // return zero, a table of width 0, which meets no band)
        const __amdgpu_buffer_rsrc_t rs_d = table_rsrc(A.vmeta + v0, nv * 16u);
        const __amdgpu_buffer_rsrc_t rs_a = table_rsrc(A.vamp + v0, nv * (unsigned)sizeof(T2));
        auto load_d = [&](unsigned b) {
            return __builtin_bit_cast(int4, __builtin_amdgcn_raw_buffer_load_b128(
                    rs_d, (int)((b + (unsigned)lane) * 16u), 0, 0));
        };
        auto load_a = [&](unsigned b) {
            return load_tap(rs_a, (b + (unsigned)lane) * (unsigned)sizeof(T2), 0u, (T2*)nullptr);
        };
        int4 d_next = load_d(0);
        T2 a_next = load_a(0);
        for (unsigned b = 0; b < nv; b += 64)
        {
            // 64 visits, one per lane: which meet the wave's cells, and from
            // where (the next 64 records are on their way meanwhile)
            const int4 d = d_next;
            const T2 a = a_next;
            d_next = load_d(b + 64);
            a_next = load_a(b + 64);
            const int W = d.w & 0xffff;
            const int top = ((d.z << 16) >> 16) - row0;      // wave's row of footprint row 0
            const int xe = (d.z >> 16) - col0;               // wave's column of unit 0
            const int skip = max(-xe, 0) / C::kUnitW;        // units left of the block
            const int xs = xe + skip * C::kUnitW;
            const int xl = min(xe + W - 1, C::kBlockW - 1);
            unsigned long long todo = __ballot(top < C::kRows && top + W > 0 && xl >= xs);
            if (!todo) continue;
            const bool mir = d.w & kBandMirror, cj = d.w & kBandConj;
            const int t0 = d.x + row0 * d.y + (mir ? -skip : skip) * C::kUnitBytes;
            // first LDS word (8: column 0), units, mirror
            const int ctl = (xs / LC + 8) | (((xl - xs) / C::kUnitW + 1) << 8) | (mir ? 1 << 12 : 0);
            const TAP ay = cj ? a.y : -a.y, aw = cj ? -a.x : a.x;

            auto visit = [&](int l, int q, auto mirrored, auto units) {
                constexpr bool MIR = decltype(mirrored)::value;
                constexpr int N = decltype(units)::value;
                const int tb = read_lane(t0, l), tp = read_lane(top, l), step = read_lane(d.y, l);
                const int w = read_lane(W, l);
                const TAP ax = read_lane(a.x, l), ays = read_lane(ay, l);
                const TAP az = read_lane(a.y, l), aws = read_lane(aw, l);
                // memory unit u holds cells' unit u, or N-1-u mirrored; rows
                // outside the footprint read zeros (out of the buffer's range)
                const int off = tb + __mul24(lr, step) +
                        (MIR ? -lane_fwd - (N - 1) * C::kUnitBytes : lane_fwd);
                const int voff = (unsigned)(lr - tp) < (unsigned)w ? off : (int)0x80000000u;
                Tap c[N];
                #pragma unroll
                for (int u = 0; u < N; ++u)
                {
                    if constexpr (C::kLaneBytes == 16)
                        c[u] = __builtin_bit_cast(Tap, __builtin_amdgcn_raw_buffer_load_b128(
                                rs_tab, voff + u * C::kUnitBytes, 0, 0));
                    else
                        c[u] = __builtin_bit_cast(Tap, __builtin_amdgcn_raw_buffer_load_b64(
                                rs_tab, voff + u * C::kUnitBytes, 0, 0));
                }
                Word* cell = cells + lane_word + (q & 255);
                Word s[N];
                #pragma unroll
                for (int u = 0; u < N; ++u) s[u] = cell[u * 8];
                #pragma unroll
                for (int u = 0; u < N; ++u)
                {
                    const Tap& k = c[MIR ? N - 1 - u : u];
                    #pragma unroll
                    for (int h = 0; h < LC; ++h)
                    {
                        const int hk = MIR ? LC - 1 - h : h;
                        const CELL cx = (CELL)k.v[2 * hk], cy = (CELL)k.v[2 * hk + 1];
                        CELL re = s[u].v[2 * h], im = s[u].v[2 * h + 1];
                        re = fma(cx, (CELL)ax, re); re = fma(cy, (CELL)ays, re);
                        im = fma(cx, (CELL)az, im); im = fma(cy, (CELL)aws, im);
                        s[u].v[2 * h] = re; s[u].v[2 * h + 1] = im;
                    }
                }
                #pragma unroll
                for (int u = 0; u < N; ++u) cell[u * 8] = s[u];
                wave_lds_fence();        // (the next visit's cells are other lanes')
            };
            auto by_units = [&](int l, int q, auto mirrored) {
                switch ((q >> 8) & 15)
                {
                case 1: visit(l, q, mirrored, std::integral_constant<int, 1>()); break;
                case 2: visit(l, q, mirrored, std::integral_constant<int, 2>()); break;
                case 3: visit(l, q, mirrored, std::integral_constant<int, 3>()); break;
                case 4: visit(l, q, mirrored, std::integral_constant<int, 4>()); break;
                case 5: visit(l, q, mirrored, std::integral_constant<int, 5>()); break;
                case 6: visit(l, q, mirrored, std::integral_constant<int, 6>()); break;
                case 7: visit(l, q, mirrored, std::integral_constant<int, 7>()); break;
                case 8: visit(l, q, mirrored, std::integral_constant<int, 8>()); break;
                default: visit(l, q, mirrored, std::integral_constant<int, C::kMaxUnits>()); break;
                }
            };
            static_assert(C::kMaxUnits == 9, "one case per number of units");
            do
            {
                const int l = __builtin_ctzll(todo);
                todo &= todo - 1ull;
                const int q = read_lane(ctl, l);
                if (q & (1 << 12)) by_units(l, q, std::true_type());
                else by_units(l, q, std::false_type());
            } while (todo);
        }

        // Out: added to the grid (single-item regions) or stored as the
        // item's partial, which k_merge sums in item order.
        const C2* cell = reinterpret_cast<const C2*>(cells + 8);
        if (I.slot == kNoSlot)
        {
            for (int r = 0; r < C::kRows; ++r)
            {
                const int y = I.y0 + row0 + r;
                if (y >= G) break;
                #pragma unroll
                for (int c = lane; c < C::kBlockW; c += 64)
                {
                    const int xg = I.x0 + col0 + c;
                    if (xg < G)
                    {
                        T2* gp = I.grid + (size_t)y * G + xg;
                        const C2 v = cell[r * C::kStride * LC + c];
                        T2 gv = *gp;
                        gv.x = (TAP)((CELL)gv.x + v.x);
                        gv.y = (TAP)((CELL)gv.y + v.y);
                        *gp = gv;
                    }
                }
            }
        }
        else
        {
            C2* out = reinterpret_cast<C2*>(A.scratch) + (size_t)I.slot * (C::kRegionW * C::kRegionH) +
                    row0 * C::kRegionW + col0;
            for (int r = 0; r < C::kRows; ++r)
                reinterpret_cast<Word*>(out + r * C::kRegionW)[lane] = cells[8 + r * C::kStride + lane];
        }
        wave_lds_fence();
    }
}

// Records of the sorted visits (see above), from one random 32-byte read per
// visit and the region of its key.
template <typename TAP, typename CELL>
__global__ __launch_bounds__(256)
void k_gather_bands(const unsigned* __restrict__ vals, const VisRec<TAP>* __restrict__ vrec,
        const unsigned* __restrict__ keys, int key_table_bits,
        const JobDev<TAP>* __restrict__ jobs, const unsigned* __restrict__ job_tile_base,
        int num_jobs, const unsigned long long* __restrict__ d_n, int4* __restrict__ vmeta,
        typename V2<TAP>::t* __restrict__ vamp)
{
    using C = BandCfg<TAP, CELL>;
    const unsigned long long n = *d_n;
    for (unsigned long long p = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x;
            p < n; p += (unsigned long long)gridDim.x * blockDim.x)
    {
        const VisRec<TAP> rec = vrec[vals[p]];
        const int4 m = rec.meta;
        const unsigned t = keys[p] >> key_table_bits;
        const int j = find_job(job_tile_base, num_jobs, t);
        const unsigned local = t - jobs[j].tile_base;
        const int ntx = jobs[j].ntx;
        const int ty = (int)(local / (unsigned)ntx);
        const int tx = (int)(local - (unsigned)ty * ntx);
        const int s = meta_support(m.z), W = 2 * s + 1;
        const bool nu = m.z & kFlagNegU, nv = m.z & kFlagNegV;
        const int top = m.y - s - ty * C::kRegionH, xl = m.x - s - tx * C::kRegionW;
        // (a lane's two cells start at an even column: the first unit may
        // start one column left of the footprint, at a zero of the table)
        const int odd = C::kLaneCells == 2 ? xl & 1 : 0;
        const int stride = table_stride(W, C::kLaneCells);
        const int tr = nv ? W - 1 + top : -top;
        const int tc = nu ? W - C::kLaneCells + odd : -odd;
        int4 d;
        d.x = (m.w + tr * stride + tc) * C::kTapBytes;
        d.y = (nv ? -stride : stride) * C::kTapBytes;
        d.z = (int)(((unsigned)(xl - odd) << 16) | ((unsigned)top & 0xffffu));
        d.w = W | (nu ? kBandMirror : 0) | ((m.z & kFlagConj) ? kBandConj : 0);
        vmeta[p] = d;
        vamp[p] = {rec.amp.x, rec.amp.y};
    }
}

// Work items (one thread each), in the order the band kernel takes them: by
// the kernel table of their first visit, in kOrderBuckets steps, when `first`
// is given (first position of each step), so that items that run side by side
// read the same tables, which their XCDs' L2s hold (2.15M visibilities, 714
// planes: kernel 3.5 -> 3.0 ms); as they come otherwise.  The order within a
// step is left open: an item's sums and its place in the merge do not depend
// on when it runs.
constexpr int kOrderBuckets = 1024;

struct BandItemArgs
{
    const unsigned* d_num_items;
    const unsigned* item_tile; const unsigned* item_off; const unsigned* slot_off;
    const unsigned* tile_start; const unsigned* tile_end;
    const unsigned* keys;            // sorted visit keys
    unsigned override;               // item size of every job, or 0: the jobs'
    unsigned table_mask; int shift;  // (key & table_mask) >> shift: the step
    const unsigned* job_tile_base; int num_jobs; int tw, th;
};

// An item's first visit and its step.
template <typename T>
__device__ __forceinline__ unsigned first_visit(const BandItemArgs& A, const JobDev<T>& J,
        unsigned item, unsigned t, unsigned& size)
{
    size = A.override ? A.override : J.visits_per_item;
    return A.tile_start[t] + (item - A.item_off[t]) * size;
}
__device__ __forceinline__ unsigned order_step(const BandItemArgs& A, unsigned visit)
{
    return (A.keys[visit] & A.table_mask) >> A.shift;
}

template <typename T>
__global__ __launch_bounds__(256)
void k_order_count(const BandItemArgs A, const JobDev<T>* __restrict__ jobs,
        unsigned* __restrict__ count)
{
    const unsigned n = *A.d_num_items;
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    {
        const unsigned t = A.item_tile[i];
        unsigned size;
        const unsigned v = first_visit(A, jobs[find_job(A.job_tile_base, A.num_jobs, t)], i, t, size);
        atomicAdd(&count[order_step(A, v)], 1u);
    }
}

// Counts -> first positions (one workgroup of kOrderBuckets threads).
__global__ __launch_bounds__(kOrderBuckets)
void k_order_scan(unsigned* __restrict__ count)
{
    __shared__ unsigned sh[kOrderBuckets];
    const unsigned c = count[threadIdx.x];
    sh[threadIdx.x] = c;
    __syncthreads();
    for (int o = 1; o < kOrderBuckets; o <<= 1)
    {
        const unsigned y = (int)threadIdx.x >= o ? sh[threadIdx.x - o] : 0u;
        __syncthreads();
        sh[threadIdx.x] += y;
        __syncthreads();
    }
    count[threadIdx.x] = sh[threadIdx.x] - c;
}

template <typename T>
__global__ __launch_bounds__(256)
void k_band_items(const BandItemArgs A, const JobDev<T>* __restrict__ jobs,
        unsigned* __restrict__ first, BandItem<T>* __restrict__ out)
{
    const unsigned n = *A.d_num_items;
    for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    {
        const unsigned t = A.item_tile[i];
        const unsigned ioff = A.item_off[t], m = i - ioff;
        const JobDev<T>& J = jobs[find_job(A.job_tile_base, A.num_jobs, t)];
        const unsigned local = t - J.tile_base;
        const unsigned ty = local / (unsigned)J.ntx, tx = local - ty * (unsigned)J.ntx;
        BandItem<T> I;
        unsigned size;
        I.v0 = first_visit(A, J, i, t, size);
        I.nv = min(size, A.tile_end[t] - I.v0);
        I.slot = A.item_off[t + 1] - ioff == 1 ? kNoSlot : A.slot_off[t] + m;
        I.x0 = (int)tx * A.tw;
        I.y0 = (int)ty * A.th;
        I.grid_size = J.grid_size;
        I.grid = J.grid;
        out[first ? atomicAdd(&first[order_step(A, I.v0)], 1u) : i] = I;
    }
}

} // namespace gg
