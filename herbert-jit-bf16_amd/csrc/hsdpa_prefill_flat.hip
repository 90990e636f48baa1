// hsdpa_prefill_flat.hip — the causal prefill in equal shares at head
// dimension 128: the key tiles of all (head group, row group) pairs of a call form
// one sequence, and each workgroup of one round walks an equal part of it,
// whatever the row groups' lengths. Where a grid of row groups, or an even
// split of each, leaves compute units idle or waiting for the longest row
// group, the shares fill them (prefill_flat has the rule and the figures).
// Three launches like the split form's: the row maxima, P.V at the exact
// maximum, and a combine of the row groups that several workgroups share. Same
// tile walks and numerics as prefill_attn; heads per workgroup and the sink are
// arguments here, so that there is one instantiation. At D = 256 the grids that
// start every workgroup at tile 0 stay: a KV head does not fit an XCD's L2,
// which then serves the workgroups that walk the same tiles at the same time.
// The smaller head dimensions have no instantiation and are not measured this
// way; a plan whose static scratch the parts would pass is laid out without them.

#include "hsdpa_attn_kernels.h"

namespace hsdpa {

static constexpr int kFlatNW = 8;                               // waves per workgroup

// The (head group, row group) pair a position of the sequence falls in, and
// the workgroups that share it. All in 32 bits (the host checks it).
__device__ __forceinline__ uint32_t flat_prefix(const FlatShape &f, uint32_t rg)
{
    return rg * f.p0 + (kFlatNW >> f.lh) * (rg * (rg + 1) / 2);
}
__device__ __forceinline__ uint32_t flat_tiles(const FlatShape &f, uint32_t rg)
{
    return rg + 1 < f.R ? f.p0 + (rg + 1) * (kFlatNW >> f.lh) : f.last;
}
// the workgroup, of W, that walks position x
__device__ __forceinline__ uint32_t flat_wg(const FlatShape &f, uint32_t x, uint32_t W)
{
    return ((x + 1) * W - 1) / f.T;
}

// A workgroup's walk, one row group after the other: head group y, row group
// rg, its position s in the sequence, its tiles nt, of them [tb, te) here.
struct FlatWalk {
    uint32_t W, w, x, x1;
    uint32_t y, rg, s, nt, tb, te;
    __device__ __forceinline__ explicit FlatWalk(const FlatShape &f)
    {
        // consecutive shares on one XCD (workgroup i runs on XCD i % 8): they
        // walk the same KV head
        W = gridDim.x;
        w = W % 8 ? blockIdx.x : blockIdx.x % 8 * (W / 8) + blockIdx.x / 8;
        x = w * f.T / W;
        x1 = (w + 1) * f.T / W;
    }
    __device__ __forceinline__ bool next(const FlatShape &f)
    {
        if (x >= x1) return false;
        y = x / f.Th;
        const uint32_t r = x - y * f.Th;
        uint32_t lo = 0, hi = f.R - 1;                          // the last row group starting at or before r
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) / 2;
            if (flat_prefix(f, mid) <= r) lo = mid;
            else hi = mid - 1;
        }
        rg = lo;
        tb = r - flat_prefix(f, rg);
        nt = flat_tiles(f, rg);
        s = x - tb;
        te = nt - tb < x1 - x ? nt : tb + (x1 - x);
        x += te - tb;
        return true;
    }
};

// One wave's rows of a row group, and its Q.
template <int D> struct FlatRows {
    int head, nfull;
    uint64_t row, lim;
    bool rowv;
    u32x4 qb[D / 16];
    __device__ __forceinline__ FlatRows(const PrefillArgs &a, const FlatShape &f, const FlatWalk &k, int wave, int l)
    {
        const int hpw = 1 << f.lh;
        head = static_cast<int>(k.y) * hpw + (wave & (hpw - 1));
        const uint64_t r0 = static_cast<uint64_t>(k.rg) * (32 * (kFlatNW >> f.lh)) + 32 * (wave >> f.lh);
        row = r0 + (l & 31);
        rowv = row < a.rows;
        nfull = r0 < a.rows ? static_cast<int>((a.past + r0 + 1) / kKeyTile) : 0;
        lim = a.past + row;
        const uint16_t *qp = a.q + (rowv ? row : 0) * a.q_row + static_cast<uint64_t>(head) * a.q_head;
#pragma unroll
        for (int s = 0; s < D / 16; s++) qb[s] = q_chunk(load16(qp + 16 * s + 8 * (l >> 5)), rowv, q_sign(a));
    }
};

// Row maxima: smax[slot][head][row], slot the workgroup's place among those
// that share the row group.
template <int D>
__global__ __launch_bounds__(64 * kFlatNW, 1) void flat_max(PrefillArgs a, FlatShape f)
{
    __shared__ __attribute__((aligned(16))) uint16_t kb[2][kKeyTile * Pad<D>::K];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    FlatWalk k(f);
    while (k.next(f)) {
        const FlatRows<D> r(a, f, k, wave, l);
        const uint16_t *kg = a.k + static_cast<uint64_t>(r.head / a.gqa) * a.kv_stride;
        float m = max_walk<D, kFlatNW>(a, kg, kb, r.qb, r.lim, r.nfull, static_cast<int>(k.tb),
                                       static_cast<int>(k.te), tid);
        m = __builtin_fmaxf(m, __shfl_xor(m, 32));
        const uint64_t slot = k.w - flat_wg(f, k.s, k.W);
        if (r.rowv && l < 32) f.smax[(slot * f.heads + r.head) * a.rows + r.row] = m;
    }
}

// P.V: a row group walked by one workgroup is written directly; otherwise the
// workgroup leaves its part in its cells, (2 w + 1) 256 .. for a row group's
// first part (the workgroup's last), 2 w 256 .. for a later one (its first).
template <int D>
__global__ __launch_bounds__(64 * kFlatNW, 1) void flat_pv(PrefillArgs a, FlatShape f)
{
    __shared__ __attribute__((aligned(16))) uint16_t kb[2][kKeyTile * Pad<D>::K];
    __shared__ __attribute__((aligned(16))) uint16_t vb[2][kKeyTile * Pad<D>::V];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, grp = l >> 5;
    FlatWalk k(f);
    while (k.next(f)) {
        const FlatRows<D> r(a, f, k, wave, l);
        const uint64_t kv = static_cast<uint64_t>(r.head / a.gqa) * a.kv_stride;
        float m = r.rowv ? kNegInf : 0.0f;
        if (r.rowv) {
            const uint32_t slots = flat_wg(f, k.s + k.nt - 1, f.wm) - flat_wg(f, k.s, f.wm) + 1;
            for (uint32_t z = 0; z < slots; z++)
                m = __builtin_fmaxf(m, f.smax[(static_cast<uint64_t>(z) * f.heads + r.head) * a.rows + r.row]);
        }
        float ms;                                               // the scaled maximum, with the sink
        const RowExp ex = causal_exp(a, m, a.sink_on != 0, ms);
        f32x16 o[D / 32];
#pragma unroll
        for (int dt = 0; dt < D / 32; dt++) o[dt] = f32x16{};
        // the sink's exponential, once per row: in its first part
        float lsum = a.sink_on && k.tb == 0 && grp == 0 ? exp_poly(a.sink - ms) : 0.0f;
        u32x4 kr[Tile<D, 64 * kFlatNW>::kPer], vr[Tile<D, 64 * kFlatNW>::kPer];
        pv_walk<D, kFlatNW, false>(a, a.k + kv, a.v + kv, kr, vr, kb, vb, r.qb, ex, r.lim, r.nfull, static_cast<int>(k.tb),
                            static_cast<int>(k.te), tid, o, lsum);
        lsum += __shfl_xor(lsum, 32);
        if (k.tb == 0 && k.te == k.nt) {
            if (r.rowv) {
                uint16_t *op = a.out + r.row * a.out_row + static_cast<uint64_t>(r.head) * D;
                const uint16_t *gp = a.gate ? a.gate + r.row * a.gate_row + static_cast<uint64_t>(r.head) * D : nullptr;
                if (a.sink_on) store_rows<D>(o, op, gp, grp, rcp_norm{1.0f / lsum});
                else store_rows<D>(o, op, gp, grp, div_norm{lsum});
            }
        } else if (r.rowv) {
            const uint64_t cell = (2 * k.w + (k.tb == 0 ? 1 : 0)) * 256 + wave * 32 + (l & 31);
            float *op = f.so + cell * D;
#pragma unroll
            for (int dt = 0; dt < D / 32; dt++)
#pragma unroll
                for (int c = 0; c < 4; c++)
                    *reinterpret_cast<f32x4 *>(op + 32 * dt + 8 * c + 4 * grp) =
                        f32x4{o[dt][4 * c], o[dt][4 * c + 1], o[dt][4 * c + 2], o[dt][4 * c + 3]};
            if (grp == 0) f.sl[cell] = lsum;
        }
    }
}

// The shared row groups' outputs, their parts added in key order.
template <int D>
__global__ __launch_bounds__(CombineShape<D>::THREADS) void flat_combine(PrefillArgs a, FlatShape f)
{
    constexpr int DL = CombineShape<D>::DL, CELLS = CombineShape<D>::CELLS;
    const int t = static_cast<int>(threadIdx.x) % DL;
    const uint32_t at = blockIdx.x * CELLS + threadIdx.x / DL, heads = f.heads, row = at / heads;
    if (row >= a.rows) return;
    const uint32_t head = at - row * heads, hpw = 1u << f.lh, rpw = 32 * (kFlatNW >> f.lh);
    const uint32_t rg = row / rpw, s = (head >> f.lh) * f.Th + flat_prefix(f, rg);
    const uint32_t w0 = flat_wg(f, s, f.wp), w1 = flat_wg(f, s + flat_tiles(f, rg) - 1, f.wp);
    if (w0 == w1) return;                                       // written directly
    const uint32_t unit = row % rpw / 32 * hpw + (head & (hpw - 1));
    f32x4 o = {};
    float L = 0.0f;
    for (uint32_t w = w0; w <= w1; w++) {
        const uint64_t cell = static_cast<uint64_t>(2 * w + (w == w0 ? 1 : 0)) * 256 + unit * 32 + row % 32;
        o += *reinterpret_cast<const f32x4 *>(f.so + cell * D + 4 * t);
        L += f.sl[cell];
    }
    combine_store<D>(a, row, head, t, o, L);
}

hipError_t launch_prefill_flat(const PrefillArgs &a, const FlatShape &f, hipStream_t s)
{
    constexpr int D = kFlatDim, CELLS = CombineShape<D>::CELLS;
    hipError_t e = launch(flat_max<D>, dim3(f.wm), dim3(64 * kFlatNW), s, a, f);
    if (e == hipSuccess) e = launch(flat_pv<D>, dim3(f.wp), dim3(64 * kFlatNW), s, a, f);
    if (e != hipSuccess) return e;
    const uint64_t cells = a.rows * f.heads;
    return launch(flat_combine<D>, dim3(static_cast<unsigned>((cells + CELLS - 1) / CELLS)),
                  dim3(CombineShape<D>::THREADS), s, a, f);
}

}  // namespace hsdpa
