// Device-side preparation of a batch: base encoding, per-read bins and a
// counting sort of all alignments into a work list ordered by (bin,
// descending hap length).
//
// Replaces the reference's convert_DNA / partitionIndicesKernel /
// computeAlignmentsPerPartitionPerBatch plus its thrust/cub scans and the
// per-chunk host round trip (utility_kernels.cuh:6-102; gpuworker.cuh:747-888).
// The reference partitions reads by the smallest tile that holds them; here a
// bin is (tile class, arithmetic form), and alignments inside a bin are
// ordered by hap length so the groups of one wave sweep the same number of
// columns.  Within a record, every alignment of a hap shares the hap's
// length, so counts and positions are reserved per (hap, bin) and the
// atomics scale with haps x bins, not alignments.
//
// Views passed here are self-contained: reads_prefix[0] == 0,
// haps_prefix[0] == 0, and read/hap offsets index read_data/hap_data.
#include "phmm_device.hpp"

namespace phmm {

// Counter arrays that k_prep zeroes (in a kernel rather than by memsets, so
// the sequence can be captured and replayed as a graph).
struct ClearList {
    int32_t* p[7];
    int32_t n[7];
    int32_t count;
};
__device__ __forceinline__ void clear_list(const ClearList& cl, int block, int nblocks)
{
    const int64_t stride = (int64_t)nblocks * blockDim.x;
    for (int k = 0; k < cl.count; ++k)
        for (int64_t i = block * (int64_t)blockDim.x + threadIdx.x; i < cl.n[k]; i += stride)
            cl.p[k][i] = 0;
}

// Grid-stride loops throughout: a launch covers any batch size, so the
// same grids serve every call when the sequence is captured in a graph.
#define GRID_STRIDE(i, n)                                                              \
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < (int64_t)(n); \
         i += (int64_t)gridDim.x * blockDim.x)

// Sequence bytes are padded to multiples of 4 per read/hap (the reference's
// padding rule) and start 4-byte aligned, so both passes below load and
// encode 4 bytes per lane: dword loads of each input array.

// One wave per hap: its code bytes (dwords over the padded length), whether
// it holds, within its length, the wildcard (reference GPU semantics: any
// byte other than A/C/G/T; CPU semantics: 'N') or, under CPU semantics, a
// byte that matches nothing but itself -- alignments with such haps go to the
// wildcard and exact bins, so the tile kernels' emission tables need only the
// four bases -- and the longest hap (per-block maxima into kHmaxParts
// counters, folded by k_scan_bins).
// Block `block` of `nblocks` (256 threads); returns its longest hap (thread 0).
__device__ __forceinline__ int hap_pass(const BinParams& bp, const BatchDesc& b, int block,
                                        int nblocks)
{
    __shared__ int wmax[4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int nwaves = nblocks * (blockDim.x >> 6);
    const uint32_t* hd = reinterpret_cast<const uint32_t*>(b.hap_data);
    uint32_t* out = reinterpret_cast<uint32_t*>(bp.hapc);
    int m = 0;
    const int h0 = block * (blockDim.x >> 6) + wv;
    // the next hap's length and offset are loaded one hap ahead
    int hl_next = h0 < b.nH ? b.hap_len[h0] : 0;
    int off_next = h0 < b.nH ? b.hap_off[h0] : 0;
    for (int h = h0; h < b.nH; h += nwaves) {
        const int hl = hl_next, d0 = off_next >> 2;
        if (h + nwaves < b.nH) {
            hl_next = b.hap_len[h + nwaves];
            off_next = b.hap_off[h + nwaves];
        }
        m = max(m, hl);
        const int nd = (max(hl, 0) >> 2) + 1;  // padded length: hl + 4 - hl % 4
        bool wild = false, exotic = false;
        for (int d = lane; d < nd; d += 64) {
            const uint32_t w = hd[d0 + d];
            uint32_t c = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                // (the padding's bytes, whatever they are, become base 0)
                const uint32_t code =
                    4 * d + k < hl ? (uint32_t)base_code_sem((uint8_t)(w >> (8 * k)), bp.semantics) : 0u;
                c |= code << (8 * k);
                wild = wild | (code == 4u);
                exotic = exotic | (code > 4u);
            }
            out[d0 + d] = c;
        }
        wild = __any(wild);
        exotic = __any(exotic);
        if (lane == 0)
            bp.hapflag[h] = exotic ? 2 : wild ? 1 : 0;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        m = max(m, __shfl_xor(m, o, 64));
    if (lane == 0)
        wmax[wv] = m;
    __syncthreads();
    int bm = 0;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k)
        bm = max(bm, wmax[k]);
    return bm;
}

// Per read (16 lanes each, four reads per wave): its packed rows and its
// bin.  Lane sl of a read's slot takes rows 4d .. 4d+3 for d = sl, sl+16,
// ... over the read's padded length: one dword of each input array, one
// 16-byte store of the packed words (base code | base q << 8 | ins q << 16 |
// del q << 24, qualities clamped to 127).  Tile class k is the first table
// row whose max_read_len covers the read (its tile has room for one more
// row); reads beyond the last row go to the multi-tile bin 2*ntiles.  Bin 2k
// uses the rescaled (FAST) arithmetic when the read's coefficients keep it in
// range, else bin 2k+1 (SAFE; a multi-tile read's form is the sign of its
// nl); under per-position gcp every row's eps enters the check.  Reference CPU
// and per-position gcp semantics: a read holding a byte other than A/C/G/T/N
// goes to the exact bin 2*ntiles+1.  The slot combines its lanes' verdicts and
// the product of alpha with row-local reductions.
// Block `block` of `nblocks` (256 threads).
__device__ __forceinline__ void read_meta(const BinParams& bp, const BatchDesc& b, int block,
                                          int nblocks)
{
    __shared__ float ph2pr[128];
    for (int q = threadIdx.x; q < 128; q += blockDim.x)
        ph2pr[q] = bp.ph2pr[q];
    __syncthreads();
    const uint32_t* rd = reinterpret_cast<const uint32_t*>(b.read_data);
    const uint32_t* q0 = reinterpret_cast<const uint32_t*>(b.bq);
    const uint32_t* q1 = reinterpret_cast<const uint32_t*>(b.iq);
    const uint32_t* q2 = reinterpret_cast<const uint32_t*>(b.dq);
    const uint32_t* q3 = reinterpret_cast<const uint32_t*>(b.gcp);
    const bool row_gcp = bp.semantics == 2;  // per-position gcp: eps of every row
    uint4* rows4 = reinterpret_cast<uint4*>(bp.rows);
    const int sl = threadIdx.x & 15;
    const int nslots = nblocks * (blockDim.x >> 4);
    // every 16-lane slot runs the same number of iterations, so the row-local
    // reductions below never have a slot missing
    const int iters = (b.nR + nslots - 1) / nslots;
    const int i0 = block * (blockDim.x >> 4) + (threadIdx.x >> 4);
    // the next read's length and offset are loaded one read ahead
    int L_next = i0 < b.nR ? b.read_len[i0] : 0;
    int off_next = i0 < b.nR ? b.read_off[i0] : 0;
    for (int it = 0; it < iters; ++it) {
        const int i = i0 + it * nslots;
        const bool valid = i < b.nR;
        const int L = valid ? L_next : 0;
        const int off_i = off_next;
        if (i + nslots < b.nR) {
            L_next = b.read_len[i + nslots];
            off_next = b.read_off[i + nslots];
        }
        int k = bp.ntiles;
        for (int j = 0; j < bp.ntiles; ++j)
            if (L <= bp.tiles[j]) {
                k = j;
                break;
            }
        const int off = (valid && L > 0) ? off_i : 0;
        const int nd = (valid && L > 0) ? (L >> 2) + 1 : 0;  // dwords of the padded read
        float eps = kEpsGpu;
        if (valid && L > 0 && bp.semantics == 1)
            eps = ph2pr[min((int)b.gcp[off], 127)];
        else if (row_gcp)
            eps = 0.f;  // the rows' own eps are checked below
        bool ok = true, exotic = false;
        double nl = 1.0;
        float pdelta = 0.f, palpha = 1.f;  // the row above this lane's first row
        // same trip count on the slot's lanes (nd is the read's)
        for (int base = 0; base < nd; base += 16) {
            const int d = base + sl;
            uint32_t w[4] = {0u, 0u, 0u, 0u};
            uint32_t gw = 0u;  // gcp bytes of the four rows (per-position gcp only)
            if (d < nd) {
                const int q = (off >> 2) + d;
                const uint32_t r = rd[q], a = q0[q], c = q1[q], e = q2[q];
                if (row_gcp)
                    gw = q3[q];
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const uint32_t code = (uint32_t)base_code_sem((uint8_t)(r >> (8 * x)), bp.semantics);
                    const uint32_t qb = min((a >> (8 * x)) & 0xffu, 127u);
                    const uint32_t qi = min((c >> (8 * x)) & 0xffu, 127u);
                    const uint32_t qd = min((e >> (8 * x)) & 0xffu, 127u);
                    w[x] = code | (qb << 8) | (qi << 16) | (qd << 24);
                }
                rows4[q] = make_uint4(w[0], w[1], w[2], w[3]);
            }
            float dl[4], al[4], sg[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                dl[x] = ph2pr[row_iq(w[x])];
                sg[x] = ph2pr[row_dq(w[x])];
                al[x] = 1.0f - (dl[x] + sg[x]);
            }
            // row 4d-1: the next lower lane's last row; lane 0 keeps the
            // previous step's lane 15 row
            const float up_delta = __shfl_up(dl[3], 1, 16);
            const float up_alpha = __shfl_up(al[3], 1, 16);
            if (sl > 0) {
                pdelta = up_delta;
                palpha = up_alpha;
            }
            // branch-free per row (bitwise logic and selects: no divergent
            // control flow inside the slot)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const int r = 4 * d + x;
                const bool in = r < L;
                // the row's gap continuation (per-position gcp: its own, at most 1/2)
                const float er = row_gcp ? ph2pr[min((gw >> (8 * x)) & 0xffu, 127u)] : eps;
                const bool range_bad = !((al[x] > 0.f) & (al[x] <= 1.f) & (dl[x] > 0.f) &
                                         (sg[x] > 0.f) & (er <= 0.5f));
                // e_r = eps_r*delta_{r-1} / (delta_r*alpha_{r-1}) > 1/2
                const bool er_bad = (r > 0) & !(er * pdelta <= 0.5f * (dl[x] * palpha));
                ok = ok & !(in & (range_bad | er_bad));
                exotic = exotic | (in & (row_code(w[x]) == kExoticCode));
                nl *= in ? (double)al[x] : 1.0;
                pdelta = dl[x];
                palpha = al[x];
            }
            const float last_delta = __shfl(dl[3], 15, 16);
            const float last_alpha = __shfl(al[3], 15, 16);
            if (sl == 0) {
                pdelta = last_delta;
                palpha = last_alpha;
            }
        }
        // reductions over the 16 lanes of this read (xor offsets < 16 stay
        // inside the 16-lane slot)
        int okv = ok ? 1 : 0, exv = exotic ? 1 : 0;
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
            nl *= __shfl_xor(nl, o, 64);
            okv &= __shfl_xor(okv, o, 64);
            exv |= __shfl_xor(exv, o, 64);
        }
        if (!valid || sl != 0)
            continue;
        ReadMeta m;
        m.nl = 1.0f;
        if (L <= 0) {
            m.bin = -1;
        } else if (bp.semantics != 0 && exv) {
            m.bin = 2 * bp.ntiles + 1;
        } else {
            bool fast = okv && bp.allow_fast != 0 && eps <= 0.5f;
            if (fast && !(nl >= 1e-30))  // the start constant must stay a normal float
                fast = false;
            const bool multi = k == bp.ntiles;
            m.nl = fast ? (float)nl : multi ? -1.0f : 1.0f;
            m.bin = multi ? 2 * k : 2 * k + (fast ? 0 : 1);
        }
        bp.meta[i] = m;
    }
}

// Exclusive prefix of R_g*H_g (the reference's resultOffsetsPerBatch,
// gpuworker.cuh:802-815), one block, 16 consecutive groups per thread
// and pass.
__device__ __forceinline__ void align_offsets(const BinParams& bp, const BatchDesc& b)
{
    constexpr int kPer = 16;
    const int G = b.G, nt = blockDim.x, nwv = nt >> 6;
    __shared__ int64_t wsum[16];
    __shared__ int64_t carry;
    if (threadIdx.x == 0)
        carry = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int base = 0; base < G; base += kPer * nt) {
        const int g0 = base + kPer * (int)threadIdx.x;
        int64_t p[kPer];
#pragma unroll
        for (int u = 0; u < kPer; ++u)
            p[u] = g0 + u < G ? (int64_t)b.nreads[g0 + u] * b.nhaps[g0 + u] : 0;
        int64_t v = 0;
#pragma unroll
        for (int u = 0; u < kPer; ++u)
            v += p[u];
        int64_t x = v;
        for (int o = 1; o < 64; o <<= 1) {
            const int64_t y = __shfl_up(x, o, 64);
            if (lane >= o)
                x += y;
        }
        if (lane == 63)
            wsum[wv] = x;
        __syncthreads();
        if (threadIdx.x == 0) {
            int64_t s = 0;
            for (int k = 0; k < nwv; ++k) {
                const int64_t t = wsum[k];
                wsum[k] = s;
                s += t;
            }
        }
        __syncthreads();
        const int64_t incl = x + wsum[wv] + carry;
        int64_t run = incl - v;
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            if (g0 + u < G)
                bp.align_off[g0 + u] = run;
            run += p[u];
        }
        __syncthreads();
        if ((int)threadIdx.x == nt - 1)
            carry = incl;
        __syncthreads();
    }
    if (threadIdx.x == 0)
        bp.align_off[G] = carry;
}

// Counters, haps, reads and alignment offsets side by side: none of them needs
// another's result.  Block 0 forms the offsets (a serial chain over the
// records), the next nclear blocks clear, nhap blocks take the haps (one
// maximum each) and the rest the reads, by far the longest.  As four launches
// in turn: 156 us for 10,000 records of 25 reads of 150 bases, 60 us for 1,000.
__global__ __launch_bounds__(256) void k_prep(BinParams bp, ClearList cl, int nclear, int nhap)
{
    const BatchDesc b = *bp.bd;
    int block = blockIdx.x;
    if (block == 0) {
        for (int q = nhap + (int)threadIdx.x; q < kHmaxParts; q += blockDim.x)
            bp.hmax_part[q] = 0;
        align_offsets(bp, b);
        return;
    }
    block -= 1;
    if (block < nclear) {
        clear_list(cl, block, nclear);
        return;
    }
    block -= nclear;
    if (block < nhap) {
        const int bm = hap_pass(bp, b, block, nhap);
        if (threadIdx.x == 0)
            bp.hmax_part[block] = bm;
        return;
    }
    read_meta(bp, b, block - nhap, (int)gridDim.x - 1 - nclear - nhap);
}

// Sort key of a unit of group g: bin, then descending hap length (or
// segment columns), then g's part -- the part only spreads the atomics of
// many groups on one length over kKeyParts counters.
__device__ __forceinline__ int key_of(int bin, int hl, int g)
{
    return bin * kKeysPerBin + (kHapBuckets - 1 - hap_bucket(hl)) * kKeyParts + (g & (kKeyParts - 1));
}

// A group's non-empty read bins (including the empty-read slot NB) in LDS:
// bin id, count and start in the group's read_perm.  Every wave of the
// block runs the build (a block of several waves writes the same values).
struct GroupBins {
    int n;
    int k[kMaxBins + 1], cnt[kMaxBins + 1], st[kMaxBins + 1];
};
__device__ __forceinline__ void group_bins_compact(const BinParams& bp, int g, GroupBins& gb)
{
    const int lane = threadIdx.x & 63;
    const int NB1 = bp.NB + 1;
    if (lane == 0)
        gb.n = 0;
    __syncthreads();
    for (int k0 = 0; k0 < NB1; k0 += 64) {  // same trip count on every lane
        const int k = k0 + lane;
        const int c = k < NB1 ? bp.gb_count[(int64_t)g * NB1 + k] : 0;
        const unsigned long long m = __ballot(c > 0);
        const int before = __popcll(m & ((1ull << lane) - 1ull));
        const int base = gb.n;
        if (c > 0) {
            gb.k[base + before] = k;
            gb.cnt[base + before] = c;
            gb.st[base + before] = bp.gb_start[(int64_t)g * NB1 + k];
        }
        __syncthreads();
        if (lane == 0)
            gb.n = base + __popcll(m);
        __syncthreads();
    }
}

// The block of a group: count the group's reads per bin (slot NB: empty
// reads), store the counts, starts and the bin-ordered read permutation for
// the scatter, and keep the non-empty bins in LDS (as group_bins_compact
// would read them back).
__device__ __forceinline__ void group_bins_build(const BinParams& bp, const BatchDesc& b, int g,
                                                 GroupBins& gb, int* cnt, int* pos)
{
    const int tid = threadIdx.x, nt = blockDim.x;
    const int NB1 = bp.NB + 1;
    for (int k = tid; k < NB1; k += nt)
        cnt[k] = 0;
    __syncthreads();
    const int r0 = b.rprefix[g], nr = b.nreads[g];
    for (int r = tid; r < nr; r += nt) {
        const int k = bp.meta[r0 + r].bin;
        atomicAdd(&cnt[k < 0 ? bp.NB : k], 1);
    }
    __syncthreads();
    if (tid == 0) {
        int s = 0, n = 0;
        for (int k = 0; k < NB1; ++k) {
            const int c = cnt[k];
            pos[k] = s;
            bp.gb_start[(int64_t)g * NB1 + k] = s;
            bp.gb_count[(int64_t)g * NB1 + k] = c;
            if (c > 0) {
                gb.k[n] = k;
                gb.cnt[n] = c;
                gb.st[n] = s;
                ++n;
            }
            s += c;
        }
        gb.n = n;
    }
    __syncthreads();
    for (int r = tid; r < nr; r += nt) {
        const int k = bp.meta[r0 + r].bin;
        const int at = atomicAdd(&pos[k < 0 ? bp.NB : k], 1);
        bp.read_perm[r0 + at] = r0 + r;
    }
    __syncthreads();
}

// Per-group hap summary, uniform across the block (every wave computes it
// and writes the same values): haps with a sequence, those of them that hold
// the wildcard and those with other bytes (hapflag 1 and 2); the rest are
// cut, in order, into segments of at most `budget` columns (at least one hap
// each) -- the super-tasks' hap ranges and their work (sort key).
constexpr int kMaxSegs = 128;
struct GroupHaps {
    int nonempty, wild, exotic, nseg;
    int hs[kMaxSegs], he[kMaxSegs], work[kMaxSegs];
    int cols[64];         // staging: columns of 64 haps (0: not cut into segments)
    uint32_t info[kMaxSegs];  // haps < kMaxSegs: hap_word
};
// Length (<= 0: empty) and flag of record hap h, from the LDS copy where
// group_haps made one.
__device__ __forceinline__ void hap_info(const BinParams& bp, const BatchDesc& b,
                                         const GroupHaps& gh, int h0, int h, int& hl, int& flag)
{
    if (h < kMaxSegs) {
        const uint32_t v = gh.info[h];
        hl = hap_word_len(v);
        flag = hap_word_flagged(v) ? bp.hapflag[h0 + h] : 0;
    } else {
        hl = b.hap_len[h0 + h];
        flag = bp.hapflag[h0 + h];
    }
}
__device__ __forceinline__ void group_haps(const BinParams& bp, const BatchDesc& b, int h0, int nh,
                                           GroupHaps& gh)
{
    int ne = 0, wi = 0, ex = 0, tot = 0;
    for (int h = (int)(threadIdx.x & 63); h < nh; h += 64) {
        const int hl = b.hap_len[h0 + h];
        if (hl > 0) {
            ++ne;
            const int flag = bp.hapflag[h0 + h];
            if (flag == 0)
                tot += hl;
            else if (flag == 1)
                ++wi;
            else
                ++ex;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ne += __shfl_xor(ne, o, 64);
        wi += __shfl_xor(wi, o, 64);
        ex += __shfl_xor(ex, o, 64);
        tot += __shfl_xor(tot, o, 64);
    }
    // greedy segments number at most 2*tot/budget + 1: a larger budget where
    // they would not fit the table
    const int budget = max(b.col_budget, (2 * tot + kMaxSegs - 2) / (kMaxSegs - 1));
    // lane 0 cuts greedily over haps staged 64 at a time in LDS (one
    // parallel load per chunk instead of a serial chain of global loads)
    int n = 0, cur = 0, start = 0;
    for (int c0 = 0; c0 < nh; c0 += 64) {
        const int h = c0 + (int)(threadIdx.x & 63);
        int cols = 0;
        if (h < nh) {
            const int hl = b.hap_len[h0 + h];
            const int flag = hl > 0 ? bp.hapflag[h0 + h] : 0;
            cols = (hl > 0 && flag == 0) ? hl : 0;
            if (h < kMaxSegs)
                gh.info[h] = hap_word(hl, flag);
        }
        gh.cols[threadIdx.x & 63] = cols;
        __syncthreads();
        if ((threadIdx.x & 63) == 0) {
            for (int i = 0; i < min(64, nh - c0); ++i) {
                const int hl = gh.cols[i];
                if (hl == 0)
                    continue;
                if (cur > 0 && cur + hl > budget) {
                    gh.hs[n] = start;
                    gh.he[n] = c0 + i;
                    gh.work[n] = cur;
                    ++n;
                    cur = 0;
                }
                if (cur == 0)
                    start = c0 + i;
                cur += hl;
            }
        }
        __syncthreads();
    }
    if ((threadIdx.x & 63) == 0) {
        gh.nonempty = ne;
        gh.wild = wi;
        gh.exotic = ex;
        if (cur > 0) {
            gh.hs[n] = start;
            gh.he[n] = nh;
            gh.work[n] = cur;
            ++n;
        }
        gh.nseg = n;
    }
    __syncthreads();
}

__device__ __forceinline__ bool is_tile_bin(const BinParams& bp, int k) { return k < 2 * bp.ntiles; }
// A tile bin's `reads` reads of a group split into chunks of W = 64/lanes
// reads: one super-task per full chunk and hap segment.  The n = reads % W
// reads left over become one-alignment items of the bin's item bin (packed
// W to a task across records, so no group of a wave idles for them).
struct ChunkPlan {
    int W, nfull, rem;
};
__device__ __forceinline__ ChunkPlan chunk_plan(const BinParams& bp, int k, int reads)
{
    ChunkPlan c;
    c.W = 64 / bp.lanes[k >> 1];
    c.nfull = reads / c.W;
    c.rem = reads - c.nfull * c.W;
    return c;
}
// The item bin of tile bin k (work-bin ids past the bins of alignments).
__device__ __forceinline__ int item_bin_of(const BinParams& bp, int k) { return bp.NB + k; }
// The bin of one-alignment items of reads of bin k against haps of a flag (a
// tile bin's with flag 0 are super-tasks and item-bin items instead).  The
// strips of the multi-tile bin take the wildcard themselves, and with it the
// reads of tiles (of callers' tables) that the wildcard tiles do not hold.
__device__ __forceinline__ int run_bin_of(const BinParams& bp, int k, int flag)
{
    const int mb = 2 * bp.ntiles;
    if (flag == 2)
        return mb + 1;
    return is_tile_bin(bp, k) ? (bp.tiles[k >> 1] < 64 * kWildRows ? mb + 2 : mb) : k;
}
// The sort key of such a run.
__device__ __forceinline__ int run_key_of(const BinParams& bp, int k, int flag, int hl, int g)
{
    const int rb = run_bin_of(bp, k, flag);
    if (rb != 2 * bp.ntiles + 2)
        return key_of(rb, hl, g);
    return rb * kKeysPerBin + (kHapBuckets - 1 - wild_bucket(k, hl)) * kKeyParts +
           (g & (kKeyParts - 1));
}

// Records with many (hap, bin) runs -- haps x min(reads, 64) above
// kBigGroupRuns -- are counted and scattered by a block of four waves
// (k_count_keys_t<4>, k_scatter_t<4>), the others by one wave each: one wave
// handling a large record's runs in turn is latency-bound.
constexpr int kBigGroupRuns = 512;
__device__ __forceinline__ bool big_group(const BatchDesc& b, int g)
{
    return (int64_t)b.nhaps[g] * min(b.nreads[g], 64) > kBigGroupRuns;
}

// Orders LDS traffic between the lanes of one wave (the waves of a block
// run different numbers of hap chunks, so no block barrier applies there).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Per group (NW = 1: one wave, the small groups; NW = 4: a block of four
// waves, the large ones): its reads per bin (group_bins_build), the per-bin
// alignment counts and the sort-key histogram.  A tile bin's full chunks get
// one key (bin, segment columns) per hap segment, counted in super-tasks;
// item bins, the multi-tile, exact and wildcard bins get one key (bin, hap length)
// per (hap, bin) run, counted in alignments.
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_count_keys_t(BinParams bp)
{
    const BatchDesc& b = *bp.bd;
    __shared__ GroupBins gb;
    __shared__ GroupHaps gh;
    __shared__ int cnt[kMaxBins + 1], pos[kMaxBins + 1];
    for (int g = blockIdx.x; g < b.G; g += gridDim.x) {
        if (big_group(b, g) != (NW > 1))  // uniform over the block
            continue;
        group_bins_build(bp, b, g, gb, cnt, pos);
        const int h0 = b.hprefix[g], nh = b.nhaps[g];
        group_haps(bp, b, h0, nh, gh);
        const int n = gb.n;
        // per bin entry: alignment counts, spread over kAlignParts counters
        // per bin (every group adds to its bins: one counter per bin would
        // serialize the atomics of all groups)
        const int part = g & (kAlignParts - 1);
        for (int e = threadIdx.x; e < n; e += 64 * NW) {
            const int k = gb.k[e], c = gb.cnt[e];
            if (k == bp.NB)
                continue;
            auto add = [&](int bin, int haps) {
                if (haps > 0)
                    atomicAdd(&bp.align_part[bin * kAlignParts + part], c * haps);
            };
            const int plain = gh.nonempty - gh.wild - gh.exotic;
            if (is_tile_bin(bp, k)) {
                add(k, plain);
                add(run_bin_of(bp, k, 1), gh.wild);
            } else {
                add(k, plain + gh.wild);
            }
            add(run_bin_of(bp, k, 2), gh.exotic);
        }
        // per (tile bin entry, hap segment): its super-tasks' key
        for (int x = threadIdx.x; x < n * gh.nseg; x += 64 * NW) {
            const int e = x / gh.nseg, sg = x - e * gh.nseg;
            const int k = gb.k[e];
            if (k != bp.NB && is_tile_bin(bp, k)) {
                const ChunkPlan c = chunk_plan(bp, k, gb.cnt[e]);
                if (c.nfull > 0)
                    atomicAdd(&bp.key_count[key_of(k, gh.work[sg], g)], c.nfull);
            }
        }
        // per (hap, bin) item run: the one-wave bins' alignments, and a tile
        // bin's left-over reads against each of its haps
        for (int x = threadIdx.x; x < nh * n; x += 64 * NW) {
            const int h = x / n, e = x - h * n;
            const int k = gb.k[e];
            int hl, flag;
            hap_info(bp, b, gh, h0, h, hl, flag);
            if (hl <= 0 || k == bp.NB)
                continue;
            if (is_tile_bin(bp, k) && flag == 0) {
                const ChunkPlan c = chunk_plan(bp, k, gb.cnt[e]);
                if (c.rem > 0)
                    atomicAdd(&bp.key_count[key_of(item_bin_of(bp, k), hl, g)], c.rem);
                continue;
            }
            atomicAdd(&bp.key_count[run_key_of(bp, k, flag, hl, g)], gb.cnt[e]);
            if (run_bin_of(bp, k, flag) == 2 * bp.ntiles)
                atomicMax(bp.strip_hmax, b.hap_len[h0 + h]);
        }
        __syncthreads();
    }
}

// Exclusive scan of each bin's key histogram (one block per bin): a thread
// per hap-length bucket adds the bucket's kKeyParts counters, the block scans
// the buckets, and each counter's cursor is its bucket's start plus the
// counters before it in the bucket.  key_cursor holds positions relative to
// the bin's begin, the bin's count goes to bin_range[2*bin+1].
__global__ __launch_bounds__(1024) void k_scan_keys(BinParams bp)
{
    static_assert(kKeyParts % 4 == 0, "buckets load as int4");
    static_assert(kAlignParts <= 1024, "one part per thread");
    __shared__ int wsum[16];
    __shared__ int carry;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int bin = blockIdx.x; bin < bp.NW; bin += gridDim.x) {
        if (bin < bp.NB) {  // fold the bin's alignment-count parts into part 0
            int v = (int)threadIdx.x < kAlignParts ? bp.align_part[bin * kAlignParts + threadIdx.x] : 0;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
                v += __shfl_xor(v, o, 64);
            if (lane == 0)
                wsum[wv] = v;
            __syncthreads();
            if (threadIdx.x == 0) {
                int t = 0;
                for (int k = 0; k < 16; ++k)
                    t += wsum[k];
                bp.align_part[bin * kAlignParts] = t;
            }
            __syncthreads();
        }
        if (threadIdx.x == 0)
            carry = 0;
        __syncthreads();
        const int base0 = bin * kKeysPerBin;
        for (int base = 0; base < kHapBuckets; base += 1024) {
            const int bk = base + threadIdx.x;
            int c[kKeyParts];
            int v = 0;
#pragma unroll
            for (int q = 0; q < kKeyParts / 4; ++q) {
                int4 x = make_int4(0, 0, 0, 0);
                if (bk < kHapBuckets)
                    x = reinterpret_cast<const int4*>(bp.key_count + base0 + bk * kKeyParts)[q];
                c[4 * q] = x.x;
                c[4 * q + 1] = x.y;
                c[4 * q + 2] = x.z;
                c[4 * q + 3] = x.w;
                v += x.x + x.y + x.z + x.w;
            }
            int x = v;
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o, 64);
                if (lane >= o)
                    x += y;
            }
            if (lane == 63)
                wsum[wv] = x;
            __syncthreads();
            if (threadIdx.x == 0) {
                int s = 0;
                for (int k = 0; k < 16; ++k) {
                    const int t = wsum[k];
                    wsum[k] = s;
                    s += t;
                }
            }
            __syncthreads();
            const int incl = x + wsum[wv] + carry;
            if (bk < kHapBuckets) {
                int run = incl - v;
#pragma unroll
                for (int q = 0; q < kKeyParts / 4; ++q) {
                    int4 y;
                    y.x = run;
                    run += c[4 * q];
                    y.y = run;
                    run += c[4 * q + 1];
                    y.z = run;
                    run += c[4 * q + 2];
                    y.w = run;
                    run += c[4 * q + 3];
                    reinterpret_cast<int4*>(bp.key_cursor + base0 + bk * kKeyParts)[q] = y;
                }
            }
            __syncthreads();
            if (threadIdx.x == 1023)
                carry = incl;
            __syncthreads();
        }
        if (threadIdx.x == 0)
            bp.bin_range[2 * bin + 1] = carry;
        __syncthreads();
    }
}

// Bin begins: exclusive scans of the bin counts -- in work units
// (bin_range, every work bin) and in alignments (align_range, the bins of
// reads) -- one wave.
// Counts come from range[2k+1], or from cnt[k] (then also stored there).
__device__ __forceinline__ void scan_pairs(int32_t* range, int NB, const int* cnt)
{
    int carry = 0;
    for (int base = 0; base < NB; base += 64) {
        const int k = base + (int)threadIdx.x;
        const int v = k < NB ? (cnt ? cnt[k] : range[2 * k + 1]) : 0;
        int x = v;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if ((int)threadIdx.x >= o)
                x += y;
        }
        if (k < NB) {
            range[2 * k] = carry + x - v;
            if (cnt)
                range[2 * k + 1] = v;
        }
        carry += __shfl(x, 63, 64);
    }
}

__global__ __launch_bounds__(64) void k_scan_bins(BinParams bp)
{
    __shared__ int tot[kMaxBins];
    {  // the longest hap, from the hap pass's per-block maxima
        int m = 0;
#pragma unroll
        for (int q = threadIdx.x; q < kHmaxParts; q += 64)
            m = max(m, bp.hmax_part[q]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            m = max(m, __shfl_xor(m, o, 64));
        if (threadIdx.x == 0)
            *bp.hmax = m;
    }
    scan_pairs(bp.bin_range, bp.NW, nullptr);
    // each bin's alignment count (k_scan_keys folded the bin's parts into
    // part 0)
    for (int k = threadIdx.x; k < bp.NB; k += 64)
        tot[k] = bp.align_part[k * kAlignParts];
    __syncthreads();
    scan_pairs(bp.align_range, bp.NB, tot);
}

// One group's item runs of haps [hc, hc + hcn) (at most kRuns (hap, bin
// entry) pairs), written by one wave: lanes reserve the runs -- tile-bin
// pairs are covered by super-tasks -- and list the others compactly; then
// the wave writes each listed run, lanes over the run's reads.  Alignments
// with an empty read or hap get -inf directly (align_host returns
// log10(0) - log10(c) for them).
template <int kRuns, bool kWaveSync>
__device__ __forceinline__ void scatter_hap_chunk(const BinParams& bp, const BatchDesc& b,
                                                  const GroupBins& gb, const GroupHaps& gh, int g,
                                                  int r0, int h0, int nh, int64_t A, int hc,
                                                  int hcn, int* run_x, int* run_base, int* w_off,
                                                  int* w_st, int* w_h, int* w_base)
{
    constexpr int kSkip = -2;  // run covered by a super-task
    const int lane = threadIdx.x & 63;
    const int n = gb.n;
    auto sync = [] {
        if (kWaveSync)
            wave_sync();
        else
            __syncthreads();
    };
    int nrun = 0;  // uniform
    for (int x0 = 0; x0 < hcn * n; x0 += 64) {  // same trip count on every lane
        const int x = x0 + lane;
        int base = kSkip;
        if (x < hcn * n) {
            const int h = hc + x / n, e = x % n;
            const int k = gb.k[e];
            int hl, flag;
            hap_info(bp, b, gh, h0, h, hl, flag);
            base = -1;  // -inf
            if (hl > 0 && k != bp.NB) {
                if (is_tile_bin(bp, k) && flag == 0) {
                    // super-tasks cover the full chunks; left-over reads
                    // become items of the bin's item bin
                    const ChunkPlan cp = chunk_plan(bp, k, gb.cnt[e]);
                    const int kb = item_bin_of(bp, k);
                    base = cp.rem == 0 ? kSkip
                                       : bp.bin_range[2 * kb] +
                                             atomicAdd(&bp.key_cursor[key_of(kb, hl, g)], cp.rem);
                } else {
                    base = bp.bin_range[2 * run_bin_of(bp, k, flag)] +
                           atomicAdd(&bp.key_cursor[run_key_of(bp, k, flag, hl, g)], gb.cnt[e]);
                }
            }
        }
        const bool keep = base != kSkip;
        const unsigned long long m = __ballot(keep);
        if (keep) {
            const int pos = nrun + __popcll(m & ((1ull << lane) - 1ull));
            run_x[pos] = x;
            run_base[pos] = base;
        }
        nrun += __popcll(m);
    }
    sync();
    // write the listed runs 64 at a time, lanes over the runs' (run, read)
    // pairs: many runs are a read or two (left-over reads), and every pair
    // costs a dependent load of read_perm
    for (int q0 = 0; q0 < nrun; q0 += 64) {  // same trip count on every lane
        const int q = q0 + lane;
        int cnt = 0, st = 0, h = 0, base = 0;
        if (q < nrun) {
            const int x = run_x[q];
            const int e = x % n;
            h = hc + x / n;
            base = run_base[q];
            cnt = gb.cnt[e];
            st = gb.st[e];
            if (base >= 0 && is_tile_bin(bp, gb.k[e])) {
                int hl, flag;
                hap_info(bp, b, gh, h0, h, hl, flag);
                if (flag == 0) {  // an item-bin run: the left-over reads only
                    const ChunkPlan cp = chunk_plan(bp, gb.k[e], cnt);
                    st += cp.nfull * cp.W;
                    cnt = cp.rem;
                }
            }
        }
        int incl = cnt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o)
                incl += y;
        }
        const int total = __shfl(incl, 63, 64);
        w_off[lane] = incl - cnt;
        w_st[lane] = st;
        w_h[lane] = h;
        w_base[lane] = base;
        sync();
        const int last = min(64, nrun - q0) - 1;
        for (int f = lane; f < total; f += 64) {
            int lo = 0, hi = last;  // the last run whose offset is <= f
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (w_off[mid] <= f)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            const int j = f - w_off[lo];
            const int rd = bp.read_perm[r0 + w_st[lo] + j];
            const int64_t out = A + (int64_t)(rd - r0) * nh + w_h[lo];
            if (w_base[lo] < 0) {
                b.scores[out] = -INFINITY;  // empty read or empty hap
            } else {
                WorkItem it;
                it.read = rd;
                it.hap = h0 + w_h[lo];
                it.out = (int32_t)out;
                it.pad = 0;
                bp.items[w_base[lo] + j] = it;
            }
        }
        sync();
    }
    sync();
}

// Write the work lists, per group.  Tile bins: the group's reads of the bin
// in full chunks of 64/lanes, one super-task per chunk and hap segment; the
// reads left over go to the bin's item bin.  Item bins, the multi-tile and
// the exact bins: one item per alignment, reserved per (hap, bin) run (haps
// in chunks that fit the LDS table).  NW = 1: one wave per group, the
// small groups (big_group).  NW = 4: a block of four waves per group, the
// others; its waves share the super-task pairs and take the hap
// chunks in turn.  Both launches stride over all groups and skip the other
// kind.
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_scatter_t(BinParams bp)
{
    const BatchDesc& b = *bp.bd;
    constexpr int kRuns = 256;
    __shared__ GroupBins gb;
    __shared__ GroupHaps gh;
    __shared__ int run_x[NW][kRuns], run_base[NW][kRuns];
    __shared__ int w_off[NW][64], w_st[NW][64], w_h[NW][64], w_base[NW][64];
    const int wv = threadIdx.x >> 6;
    for (int g = blockIdx.x; g < b.G; g += gridDim.x) {
        if (big_group(b, g) != (NW > 1))  // uniform over the block
            continue;
        group_bins_compact(bp, g, gb);
        const int r0 = b.rprefix[g];
        const int h0 = b.hprefix[g], nh = b.nhaps[g];
        const int64_t A = bp.align_off[g];
        group_haps(bp, b, h0, nh, gh);
        const int n = gb.n;
        // super-tasks of the tile bins: read chunks x hap segments, one
        // thread per (bin entry, segment) pair: it reserves the pair's list
        // slots and writes its tasks
        const int npairs = n * gh.nseg;
        for (int x = threadIdx.x; x < npairs; x += 64 * NW) {
            const int e = x / gh.nseg, sg = x - e * gh.nseg;
            const int k = gb.k[e];
            if (k == bp.NB || !is_tile_bin(bp, k))
                continue;
            const ChunkPlan cp = chunk_plan(bp, k, gb.cnt[e]);
            SuperTask t;
            t.h0 = h0;
            t.nh = nh;
            t.hs = gh.hs[sg];
            t.r0 = r0;
            t.aoff = (int32_t)A;
            if (cp.nfull > 0) {
                const int base = bp.bin_range[2 * k] +
                                 atomicAdd(&bp.key_cursor[key_of(k, gh.work[sg], g)], cp.nfull);
                t.nc = cp.W;
                t.he = gh.he[sg];
                for (int j = 0; j < cp.nfull; ++j) {
                    t.perm = r0 + gb.st[e] + j * cp.W;
                    bp.st[base + j] = t;
                }
            }
        }
        const int hchunk = n > 0 ? max(1, kRuns / n) : nh;
        for (int hc = wv * hchunk; hc < nh; hc += NW * hchunk)
            scatter_hap_chunk<kRuns, (NW > 1)>(bp, b, gb, gh, g, r0, h0, nh, A, hc,
                                               min(hchunk, nh - hc), run_x[wv], run_base[wv],
                                               w_off[wv], w_st[wv], w_h[wv], w_base[wv]);
        __syncthreads();  // the next group rebuilds gb and gh
    }
}

// ---------------------------------------------------------------------------
// Small calls: the whole preparation in three launches
// ---------------------------------------------------------------------------
// A small call's time is its launches: each of the sequence's kernels costs
// 4.5 us by itself, the descriptor's copy with the gaps around it 23 us, and
// the counting sort's passes are latency (a record's runs in turn, atomics of
// many records on one hap length).  Its tasks need no order -- they are fewer
// than the device's waves or not many more -- so three kernels write them:
// k_tiny_desc brings the descriptor in its arguments, k_prep encodes haps
// and reads side by side, k_tiny_plan cuts one record per block into tasks.
// Before -> after, us per call: 250 reads x 32 haps 226 -> 153, 1000 records of
// 8 x 4 300 -> 128, 50 records of 8 x 4 133 -> 68.
// (The descriptor first lay in pinned memory that the kernel read, which held
// a caller back after two calls: 131 us for the 1000 records, 125 so.)
__global__ __launch_bounds__(256) void k_tiny_desc(BinParams bp, TinyLists tl, BatchDesc d,
                                                   int late_begin)
{
    const int i = threadIdx.x;
    if (i == 0)
        *const_cast<BatchDesc*>(bp.bd) = d;
    if (i < kTinyCounts)
        tl.counts[i] = 0;
    if (i < 4)
        tl.counts[kTinyFinalRange + i] = i == 2 ? late_begin : 0;
    if (i == 0)
        *bp.task_ctr = 0;
}

// A record's hap segments for k_tiny_plan (one wave): n = columns / budget of
// about equal columns, each hap in the segment that holds its middle, or one
// hap each.
__device__ __forceinline__ void tiny_haps(const BinParams& bp, const BatchDesc& b, int h0, int nh,
                                          GroupHaps& gh)
{
    const int lane = threadIdx.x & 63;
    int ne = 0, wi = 0, ex = 0, tot = 0, normal = 0;
    for (int h = lane; h < nh; h += 64) {
        const int hl = max(b.hap_len[h0 + h], 0), flag = bp.hapflag[h0 + h];
        if (h < kMaxSegs)
            gh.info[h] = hap_word(hl, flag);
        ne += hl > 0;
        wi += (hl > 0) & (flag == 1);
        ex += (hl > 0) & (flag == 2);
        normal += (hl > 0) & (flag == 0);
        tot += flag == 0 ? hl : 0;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ne += __shfl_xor(ne, o, 64);
        wi += __shfl_xor(wi, o, 64);
        ex += __shfl_xor(ex, o, 64);
        normal += __shfl_xor(normal, o, 64);
        tot += __shfl_xor(tot, o, 64);
    }
    const int want = (int)((float)tot / (float)b.col_budget + 0.5f);
    const int n = max(1, min(want, min(normal, kMaxSegs - 1)));
    // (64 bits: exact columns, so a later hap's segment is never a lower one)
    const double scale = (double)n / (double)max(tot, 1);
    const bool each = n == normal;
    int before = 0, haps = 0, segs = 0, last = -1;  // columns, haps, segments and segment so far
    for (int c0 = 0; c0 < nh; c0 += 64) {
        const int h = c0 + lane;
        int cols = 0;
        if (h < nh) {
            const int hl = b.hap_len[h0 + h];
            cols = hl > 0 && bp.hapflag[h0 + h] == 0 ? hl : 0;
        }
        int x = cols;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            x += lane >= o ? y : 0;
        }
        const int at = before + x - cols;  // columns before this hap
        const unsigned long long m = __ballot(cols > 0);
        const unsigned long long below = m & ((1ull << lane) - 1);
        const int sg = each ? haps + __popcll(below)
                            : min((int)(((double)at + 0.5 * (double)cols) * scale), n - 1);
        const int prev = __shfl(sg, below ? 63 - __clzll((long long)below) : 0, 64);
        const bool first = cols > 0 && sg != (below ? prev : last);
        const unsigned long long f = __ballot(first);
        if (first) {
            const int q = segs + __popcll(f & ((1ull << lane) - 1));
            gh.hs[q] = h;
            if (q > 0)
                gh.he[q - 1] = h;
        }
        segs += __popcll(f);
        before += __shfl(x, 63, 64);
        haps += __popcll(m);
        if (m)
            last = __shfl(sg, 63 - __clzll((long long)m), 64);
    }
    if (lane == 0) {
        gh.nonempty = ne;
        gh.wild = wi;
        gh.exotic = ex;
        gh.nseg = segs;
        if (segs > 0)
            gh.he[segs - 1] = nh;
    }
}

// Per record: its reads ordered by (form, tile class), longest first, cut into
// chunks of as many of a class as fit side by side (the last may hold fewer;
// a chunk does not go on into the next class, whose reads would sweep more
// columns past the hap than they do elsewhere, and with them the scaling's
// verdict could differ), each against the record's hap segments; and the
// items of the other bins.  A record is one block's chain of dependent steps:
// classes, haps and tasks each in parallel over lanes (28.6 us for 250 reads
// against 32 haps where one lane went over them, 8.0 now).
__global__ __launch_bounds__(256) void k_tiny_plan(BinParams bp, TinyLists tl)
{
    const BatchDesc b = *bp.bd;
    __shared__ GroupHaps gh;
    __shared__ int cnt[kMaxBins + 1], pos[kMaxBins + 1];
    // a class's chunks: reads at .. end-1, the first chunk's number, reads per
    // chunk, lanes per read
    struct Run {
        int at, end, first, W, G;
    };
    __shared__ Run runs[2][kMaxTiles];
    __shared__ int nruns[2], nchunks[2], base[2], item_base[3], item_n[3];
    static_assert(kMaxTiles <= 64, "one class per lane");
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int mb = 2 * bp.ntiles, NB1 = bp.NB + 1;
    if (blockIdx.x == 0 && tid < 64) {  // the longest hap
        int m = 0;
        for (int q = tid; q < kTinyHapBlocks; q += 64)
            m = max(m, bp.hmax_part[q]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            m = max(m, __shfl_xor(m, o, 64));
        if (tid == 0)
            *bp.hmax = m;
    }
    for (int g = blockIdx.x; g < b.G; g += gridDim.x) {
        const int r0 = b.rprefix[g], nr = b.nreads[g], h0 = b.hprefix[g], nh = b.nhaps[g];
        const int64_t A = bp.align_off[g];
        for (int k = tid; k < NB1; k += 256)
            cnt[k] = 0;
        __syncthreads();
        for (int r = tid; r < nr; r += 256) {
            const int k = bp.meta[r0 + r].bin;
            atomicAdd(&cnt[k < 0 ? bp.NB : k], 1);
        }
        if (wv == 3)
            tiny_haps(bp, b, h0, nh, gh);
        __syncthreads();
        if (wv < 2) {
            // this form's classes (form = wave), the longest first: lane l has
            // class ntiles-1-l
            const int c = bp.ntiles - 1 - lane, k = 2 * c + wv;
            const int reads = c >= 0 ? cnt[k] : 0;
            const int G = c >= 0 ? bp.lanes[c] : 64, W = 64 / G;
            const int chunks = (reads + W - 1) / W;
            int at = reads, nc = chunks;  // inclusive sums
            int fast = c >= 0 && wv == 1 ? cnt[2 * c] : 0;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(at, o, 64), z = __shfl_up(nc, o, 64);
                at += lane >= o ? y : 0;
                nc += lane >= o ? z : 0;
                fast += __shfl_xor(fast, o, 64);  // SAFE after FAST
            }
            const unsigned long long m = __ballot(reads > 0);
            if (c >= 0)
                pos[k] = fast + at - reads;
            if (reads > 0) {
                Run& r = runs[wv][__popcll(m & ((1ull << lane) - 1))];
                r.at = fast + at - reads;
                r.end = fast + at;
                r.first = nc - chunks;
                r.W = W;
                r.G = G;
            }
            if (lane == 63) {
                const int tasks = nc * gh.nseg;
                nruns[wv] = __popcll(m);
                nchunks[wv] = nc;
                base[wv] = tasks > 0 ? atomicAdd(&tl.counts[kTinyFast + wv], tasks) : 0;
            }
        } else if (wv == 2) {  // the other bins' reads, after both forms
            int at = 0;
            for (int k = lane; k < mb; k += 64)
                at += cnt[k];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
                at += __shfl_xor(at, o, 64);
            if (lane == 0)
                for (int k = mb; k < NB1; ++k) {
                    pos[k] = at;
                    at += cnt[k];
                }
        }
        __syncthreads();
        for (int r = tid; r < nr; r += 256) {
            const int k = bp.meta[r0 + r].bin;
            bp.read_perm[r0 + atomicAdd(&pos[k < 0 ? bp.NB : k], 1)] = r0 + r;
        }
        // super-tasks: a class per wave, a hap segment per lane; tasks of one
        // segment lie together, the longest class first
        for (int form = 0; form < 2; ++form) {
            const int n = nruns[form], nc = nchunks[form];
            for (int q = wv; q < n; q += 4) {
                const Run r = runs[form][q];
                const int chunks = (r.end - r.at + r.W - 1) / r.W;
                // one chunk's segments, or with few segments several chunks' at once
                const int side = max(1, min(64 / max(gh.nseg, 1), chunks));
                for (int ch0 = 0; ch0 < chunks; ch0 += side)
                    for (int y = lane; y < gh.nseg * side; y += 64) {
                        const int sg = y / side, ch = ch0 + y - sg * side;
                        if (ch >= chunks)
                            continue;
                        const int at = r.at + ch * r.W;
                        SuperTask t;
                        t.perm = r0 + at;
                        t.nc = min(r.W, r.end - at) | r.G << 8;
                        t.h0 = h0;
                        t.nh = nh;
                        t.hs = gh.hs[sg];
                        t.he = gh.he[sg];
                        t.r0 = r0;
                        t.aoff = (int32_t)A;
                        tl.st[form][base[form] + sg * nc + r.first + ch] = t;
                    }
            }
        }
        // one-alignment items (strips, wildcard, exact) and empty alignments
        const int odd = cnt[mb] + cnt[mb + 1] + cnt[mb + 2] + cnt[bp.NB];
        if (odd > 0 || gh.nonempty < nh || gh.wild + gh.exotic > 0) {  // uniform
            if (tid < 3)
                item_n[tid] = 0;
            const bool plain_haps = gh.nonempty == nh && gh.wild + gh.exotic == 0;
            int strip_h = 0;
            // two passes over the pairs, a read per wave: count, then write
            for (int pass = 0; pass < 2; ++pass) {
                __syncthreads();
                if (pass == 1 && tid < 3) {
                    item_base[tid] = item_n[tid] > 0 ? atomicAdd(&tl.counts[kTinyStrips + tid], item_n[tid]) : 0;
                    item_n[tid] = 0;
                }
                __syncthreads();
                for (int r = wv; r < nr; r += 4) {
                    const int k = bp.meta[r0 + r].bin;
                    const bool tile = k >= 0 && is_tile_bin(bp, k);
                    if (tile && plain_haps)
                        continue;
                    const int64_t row = A + (int64_t)r * nh;
                    for (int h1 = 0; h1 < nh; h1 += 64) {
                        const int h = h1 + lane;
                        int hl = 0, flag = 0;
                        if (h < nh)
                            hap_info(bp, b, gh, h0, h, hl, flag);
                        const bool empty = h < nh && (k < 0 || hl <= 0);
                        if (empty && pass == 0)
                            b.scores[row + h] = -INFINITY;
                        const bool item = h < nh && !empty && !(tile && flag == 0);
                        const int rb = item ? run_bin_of(bp, k, flag) : -1;
                        const int list = !item ? -1 : rb == mb ? 0 : rb == mb + 2 ? 1 : 2;
                        for (int l = 0; l < 3; ++l) {
                            const unsigned long long m = __ballot(list == l);
                            if (!m)
                                continue;
                            int at = 0;
                            if (lane == 0)
                                at = atomicAdd(&item_n[l], __popcll(m));
                            at = __shfl(at, 0, 64);
                            if (pass == 0 && l == 0 && list == 0)
                                strip_h = max(strip_h, b.hap_len[h0 + h]);
                            if (pass == 0 || list != l)
                                continue;
                            WorkItem it;
                            it.read = r0 + r;
                            it.hap = h0 + h;
                            it.out = (int32_t)(row + h);
                            it.pad = 0;
                            WorkItem* out = l == 0 ? tl.strips : l == 1 ? tl.wilds : tl.exact;
                            out[item_base[l] + at + __popcll(m & ((1ull << lane) - 1))] = it;
                        }
                    }
                }
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
                strip_h = max(strip_h, __shfl_xor(strip_h, o, 64));
            if (lane == 0 && strip_h > 0)
                atomicMax(bp.strip_hmax, strip_h);
        }
        __syncthreads();  // the next record rebuilds the tables
    }
}

hipError_t launch_tiny_desc(const BinParams& bp, const TinyLists& tl, const BatchDesc& d,
                            int late_begin, hipStream_t st)
{
    hipLaunchKernelGGL(k_tiny_desc, dim3(1), dim3(256), 0, st, bp, tl, d, late_begin);
    return hipGetLastError();
}

hipError_t launch_tiny_prep(const BinParams& bp, hipStream_t st)
{
    static_assert(kTinyHapBlocks <= kHmaxParts, "one maximum per block");
    hipLaunchKernelGGL(k_prep, dim3(1 + kTinyHapBlocks + kTinyReadBlocks), dim3(256), 0, st, bp,
                       ClearList{}, 0, kTinyHapBlocks);
    return hipGetLastError();
}

hipError_t launch_tiny_plan(const BinParams& bp, const TinyLists& tl, int grid, hipStream_t st)
{
    hipLaunchKernelGGL(k_tiny_plan, dim3(grid), dim3(256), 0, st, bp, tl);
    return hipGetLastError();
}

__global__ void k_add_counts(CountSums c)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        for (int k = 0; k < c.n; ++k) {
            int64_t s = 0;
            for (int i = 0; i < c.len[k]; ++i)
                s += c.counts[k][i];
            // calls on several streams may add at once
            atomicAdd(reinterpret_cast<unsigned long long*>(c.total[k]), (unsigned long long)s);
        }
    }
}

hipError_t launch_add_counts(const CountSums& c, hipStream_t st)
{
    if (c.n < 1 || c.n > CountSums::kMax)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_add_counts, dim3(1), dim3(64), 0, st, c);
    return hipGetLastError();
}

hipError_t launch_add_count(int64_t* total, const int32_t* counts, int n, hipStream_t st)
{
    CountSums c;
    c.n = 1;
    c.total[0] = total;
    c.counts[0] = counts;
    c.len[0] = n;
    return launch_add_counts(c, st);
}

// ---------------------------------------------------------------------------
hipError_t run_binning(const BinParams& bp, const BatchDesc& hd, bool fixed_grids, bool small,
                       hipStream_t st)
{
    const int tpb = 256;
    // grids: sized to the batch, or fixed (graph capture) at a size that
    // still fills the chip -- a quarter of it for the small-batch sequence,
    // whose batches are too small to use more and whose latency pays for
    // every idle wave dispatched
    auto grid = [&](int64_t n, int per_block, int cap) {
        if (fixed_grids)
            return small ? cap / 4 : cap;
        int64_t b = (n + per_block - 1) / per_block;
        return (int)(b < cap ? (b < 1 ? 1 : b) : cap);
    };
    ClearList cl{};
    cl.p[0] = bp.key_count;
    cl.n[0] = bp.NW * kKeysPerBin;
    cl.p[1] = bp.rescue_counts;
    cl.n[1] = bp.NB;
    cl.p[2] = bp.final_count;
    cl.n[2] = 1;
    cl.p[3] = bp.task_ctr;
    cl.n[3] = kTaskCounters;
    cl.p[4] = bp.align_part;
    cl.n[4] = kAlignParts * bp.NB;
    cl.p[5] = bp.retry_counts;
    cl.n[5] = kRetrySlots;
    cl.p[6] = bp.strip_hmax;
    cl.n[6] = 1;
    cl.count = 7;
    const int nclear = 64;
    const int nhap = std::min(kHmaxParts, grid(hd.nH, tpb / 64, 4096));  // one wave per hap
    const int nread = grid(hd.nR, tpb / 16, 4096);                       // 16 lanes per read
    hipLaunchKernelGGL(k_prep, dim3(1 + nclear + nhap + nread), dim3(tpb), 0, st, bp, cl, nclear, nhap);
    if (fixed_grids || hd.G > 0) {
        hipLaunchKernelGGL(k_count_keys_t<1>, dim3(grid(hd.G, 1, 8192)), dim3(64), 0, st, bp);
        hipLaunchKernelGGL(k_count_keys_t<4>, dim3(grid(hd.G, 1, 2048)), dim3(256), 0, st, bp);
    }
    hipLaunchKernelGGL(k_scan_keys, dim3(bp.NW), dim3(1024), 0, st, bp);
    hipLaunchKernelGGL(k_scan_bins, dim3(1), dim3(64), 0, st, bp);
    if (fixed_grids || hd.G > 0) {
        hipLaunchKernelGGL(k_scatter_t<1>, dim3(grid(hd.G, 1, 8192)), dim3(64), 0, st, bp);
        hipLaunchKernelGGL(k_scatter_t<4>, dim3(grid(hd.G, 1, 2048)), dim3(256), 0, st, bp);
    }
    return hipGetLastError();
}

}  // namespace phmm
