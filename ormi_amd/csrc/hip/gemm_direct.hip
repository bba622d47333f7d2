// Products that leave the tiled kernels idle: few rows or columns, small
// batches of small matrices, and operands whose rows are not whole 16-byte chunks
// (ragged extents, unaligned bases).
//
// The tiled kernels stage 128- or 256-wide tiles through LDS with direct loads
// of aligned 16-byte chunks. Here every wave loads its MFMA fragments straight
// from memory into registers, from any element address, so there is no tile to
// fill, no alignment to meet and no barrier in the main loop: a wave computes
// 16 MT x 16 NT elements over a share of K, the W waves of a work-group split K
// among them, and their partial tiles meet in LDS, where each wave adds some of
// the tile's rows in wave order, applies the epilogue and stores them. So most
// products need no workspace and no second kernel. Where the tiles leave a
// quarter of the chip idle and K is long, up to 8 work-groups share a tile's K:
// their tiles go to a workspace, and the finish pass (gemm.hip) adds them in
// split order and applies the epilogue.
//
// Fragments. A 16 x 16 MFMA takes, per lane, KV consecutive k of one row of A
// and one column of B (KV = 8 values of 16 bits, 4 floats for four K = 4
// MFMAs); lane l holds row (column) l % 16 and k-slots KV (l / 16) on. k order
// within the product is free as long as A and B agree, and so is the order of
// rows and columns as long as the store agrees:
//   k-contiguous operand: fragment f is rows 16 f + l % 16, one 16-byte load.
//   mn-contiguous operand: KV loads, one per k, of F consecutive elements at
//     F (l % 16): element j belongs to fragment j, so fragment j is rows
//     F (l % 16) + j. 16-bit values are paired by byte permutes.
// A wave's 16 lanes then read 16 F consecutive elements of each k-row: 128
// bytes at F = 4, the cache line of a weight matrix read once.
//
// What bounds it: memory for few rows (a 12 x 2048 x 8192 bf16 product reads 33
// MB of weights), fragment loads through the L1 otherwise.
#include <algorithm>
#include <type_traits>

#include "gemm_mfma.h"
#include "ormi_hip_internal.h"

namespace ormi_hip {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
// Loads at any element address.
typedef unsigned u32x4_any16 __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned u32x2_any16 __attribute__((ext_vector_type(2), aligned(2)));
typedef unsigned u32_any16 __attribute__((aligned(2)));
typedef unsigned u32x4_any32 __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned u32x2_any32 __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2_any __attribute__((ext_vector_type(2), aligned(4)));

template <typename Tr>
__device__ __forceinline__ void mma16(const u32x4_t& a, const u32x4_t& b, f32x4_t& acc) {
    if constexpr (Tr::ESIZE == 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[e]), __uint_as_float(b[e]), acc, 0, 0, 0);
    } else if constexpr (std::is_same<Tr, TrBF16>::value) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), acc, 0, 0, 0);
    } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), acc, 0, 0, 0);
    }
}

// One operand of a wave's tile: rows (of A) or columns (of B) mn0 .. mn0 + 16 F
// - 1 of MN. Rows past the end repeat valid ones and are not stored.
template <typename Tr, int F, bool KC>
struct Operand {
    static constexpr int ES = Tr::ESIZE, KV = Tr::VE, KSTEP = 4 * KV;
    struct Raw {
        unsigned r[4 * F];
    };
    const char* base;    // this lane's first element at k = 0
    long long row_step;  // KC: bytes between fragments; else bytes per k
    int first;           // mn of this lane's element in fragment 0

    // p: the operand of this batch; s_mn, s_k: its strides in elements.
    __device__ void init(const char* p, long long s_mn, long long s_k, int mn0, int MN, int lane) {
        const int c = lane & 15, g = lane >> 4;
        if constexpr (KC) {
            // Fragment f's row clamps on its own (row()).
            first = mn0 + c;
            base = p + (long long)g * KV * ES;
            row_step = s_mn * ES;
            limit = MN - 1;
        } else {
            const int start = mn0 + F * c;
            first = start < MN - F ? start : MN - F;
            base = p + ((long long)first + (long long)g * KV * s_k) * ES;
            row_step = s_k * ES;
            limit = start;  // elements before `start` repeat the previous lane's
        }
    }
    int limit;

    __device__ int row(int f) const {  // KC
        const int r = first + 16 * f;
        return r < limit ? r : limit;
    }
    // Whether element j of the tile (see mn()) is this lane's to store.
    __device__ bool owns(int f, int MN) const {
        if constexpr (KC) return first + 16 * f < MN;
        else return first + f >= limit;
    }
    // The element index fragment f's row (column) stands for.
    __device__ int mn(int f) const {
        if constexpr (KC) return first + 16 * f;
        else return first + f;
    }

    // k0: a multiple of KSTEP with k0 + KSTEP <= K.
    __device__ void load(Raw& raw, int k0) const {
        if constexpr (KC) {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const char* q = base + (long long)row(f) * row_step + (long long)k0 * ES;
                u32x4_t v;
                if constexpr (ES == 2) v = *(const u32x4_any16*)q;
                else v = *(const u32x4_any32*)q;
#pragma unroll
                for (int d = 0; d < 4; ++d) raw.r[4 * f + d] = v[d];
            }
        } else {
            const char* q = base + (long long)k0 * row_step;
#pragma unroll
            for (int e = 0; e < KV; ++e, q += row_step) {
                if constexpr (ES == 4) {
                    if constexpr (F == 4) {
                        const u32x4_t v = *(const u32x4_any32*)q;
#pragma unroll
                        for (int d = 0; d < 4; ++d) raw.r[4 * e + d] = v[d];
                    } else if constexpr (F == 2) {
                        const u32x2_any32 v = *(const u32x2_any32*)q;
                        raw.r[2 * e] = v[0];
                        raw.r[2 * e + 1] = v[1];
                    } else {
                        raw.r[e] = *(const unsigned*)q;
                    }
                } else {
                    if constexpr (F == 4) {
                        const u32x2_any16 v = *(const u32x2_any16*)q;
                        raw.r[2 * e] = v[0];
                        raw.r[2 * e + 1] = v[1];
                    } else if constexpr (F == 2) {
                        raw.r[e] = *(const u32_any16*)q;
                    } else {
                        // Two k per register.
                        const unsigned v = *(const unsigned short*)q;
                        raw.r[e / 2] = e % 2 ? raw.r[e / 2] | (v << 16) : v;
                    }
                }
            }
        }
    }

    // The last, partial k-step: elements past K are zero.
    __device__ void load_tail(Raw& raw, int k0, int K, int lane) const {
        const int kb = k0 + (lane >> 4) * KV;
#pragma unroll
        for (int d = 0; d < 4 * F; ++d) raw.r[d] = 0;
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int e = 0; e < KV; ++e) {
                if (kb + e >= K) continue;
                const char* q;
                if constexpr (KC) q = base + (long long)row(f) * row_step + (long long)(k0 + e) * ES;
                else q = base + (long long)(k0 + e) * row_step + f * ES;
                put(raw, f, e, ES == 4 ? *(const unsigned*)q : (unsigned)*(const unsigned short*)q);
            }
    }
    // Value v of fragment f, k-slot e, in the raw layout.
    __device__ static void put(Raw& raw, int f, int e, unsigned v) {
        if constexpr (ES == 4) {
            raw.r[KC ? 4 * f + e : F * e + f] = v;
        } else {
            const int at = KC ? 8 * f + e : F == 1 ? e : F * e + f;  // in 16-bit units
            raw.r[at / 2] |= v << (16 * (at % 2));
        }
    }

    __device__ static u32x4_t frag(const Raw& raw, int f) {
        if constexpr (KC || F == 1) {
            return u32x4_t{raw.r[4 * f], raw.r[4 * f + 1], raw.r[4 * f + 2], raw.r[4 * f + 3]};
        } else if constexpr (ES == 4) {
            return u32x4_t{raw.r[f], raw.r[F + f], raw.r[2 * F + f], raw.r[3 * F + f]};
        } else {
            // Halves f % 2 of the dwords that hold element f of k-rows 2d, 2d + 1.
            u32x4_t v;
#pragma unroll
            for (int d = 0; d < 4; ++d)
                v[d] = __builtin_amdgcn_perm(raw.r[(2 * d + 1) * (F / 2) + f / 2], raw.r[2 * d * (F / 2) + f / 2],
                                             f % 2 ? 0x07060302u : 0x05040100u);
            return v;
        }
    }
};

// Waves per work-group: their partial tiles take 64 KB of LDS at most.
template <int MT, int NT>
constexpr int kMostWaves = 64 / (MT * NT) < 16 ? 64 / (MT * NT) : 16;

template <typename Tr, int MT, int NT, bool A_KC, bool B_KC>
__global__ __launch_bounds__((64 * kMostWaves<MT, NT>)) void gemm_direct_kernel(GemmParams p) {
    using OA = Operand<Tr, MT, A_KC>;
    using OB = Operand<Tr, NT, B_KC>;
    constexpr int KSTEP = OA::KSTEP;
    constexpr int D = MT * NT >= 8 ? 2 : 4;  // k-steps in flight
    extern __shared__ float part[];          // the waves' partial tiles
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), W = blockDim.x >> 6;
    // Tiles of one XCD (work-groups go round them in turn) are neighbours along
    // N, so the cache lines they share stay in one L2.
    const int tiles = p.tiles_m * p.tiles_n, x = blockIdx.x & 7, q = tiles >> 3, r = tiles & 7;
    const int tile = x * q + (x < r ? x : r) + (int)(blockIdx.x >> 3);
    const int m0 = tile / p.tiles_n * 16 * MT, n0 = tile % p.tiles_n * 16 * NT;
    long long a_off = 0, b_off = 0, d_off = 0;
    const int split = blockIdx.z / p.batch;
    int bidx = blockIdx.z - split * p.batch;
    // A split's partial products lie one output apart in the workspace.
    const long long c_off = (long long)blockIdx.z * p.M * p.N;
    for (int d = p.batch_ndim - 1; d >= 0; --d) {
        const int coord = bidx % p.batch_shape[d];
        bidx /= p.batch_shape[d];
        a_off += coord * p.a_bs[d];
        b_off += coord * p.b_bs[d];
        d_off += coord * p.epi.d_bs[d];
    }
    OA oa;
    OB ob;
    oa.init(p.a + a_off * Tr::ESIZE, p.a_sm, p.a_sk, m0, p.M, lane);
    ob.init(p.b + b_off * Tr::ESIZE, p.b_sn, p.b_sk, n0, p.N, lane);

    f32x4_t acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto mma = [&](const typename OA::Raw& ra, const typename OB::Raw& rb) {
        u32x4_t fb[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) fb[j] = OB::frag(rb, j);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const u32x4_t fa = OA::frag(ra, i);
#pragma unroll
            for (int j = 0; j < NT; ++j) mma16<Tr>(fa, fb[j], acc[i][j]);
        }
    };

    // This wave's whole k-steps [s, s1): consecutive shares of the splits'
    // waves.
    const int steps = p.K / KSTEP, share = split * W + w, shares = p.splits * W;
    int s = (int)((long long)steps * share / shares);
    const int s1 = (int)((long long)steps * (share + 1) / shares);
    typename OA::Raw ra[D];
    typename OB::Raw rb[D];
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (s + d < s1) {
            oa.load(ra[d], (s + d) * KSTEP);
            ob.load(rb[d], (s + d) * KSTEP);
        }
    for (; s + 2 * D <= s1; s += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            mma(ra[d], rb[d]);
            oa.load(ra[d], (s + d + D) * KSTEP);
            ob.load(rb[d], (s + d + D) * KSTEP);
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (s + d < s1) {
            mma(ra[d], rb[d]);
            if (s + d + D < s1) {
                oa.load(ra[d], (s + d + D) * KSTEP);
                ob.load(rb[d], (s + d + D) * KSTEP);
            }
        }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (s + d + D < s1) mma(ra[d], rb[d]);
    if (share == shares - 1 && steps * KSTEP < p.K) {
        oa.load_tail(ra[0], steps * KSTEP, p.K, lane);
        ob.load_tail(rb[0], steps * KSTEP, p.K, lane);
        mma(ra[0], rb[0]);
    }

    // The waves' partial tiles meet in LDS; wave w then adds (in wave order) and
    // stores every W-th row of register groups. Accumulator register t of lane l is A's
    // fragment row 4 (l / 16) + t and B's fragment column l % 16.
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int t = 0; t < 4; ++t) part[((w * MT + i) * 4 + t) * NT * 64 + j * 64 + lane] = acc[i][j][t];
    __syncthreads();
    const Epi& e = p.epi;
    const float sv = e.s ? *e.s : 0.0f;
    float* const c = p.c + c_off;
    float* const aux = e.aux ? e.aux + c_off : nullptr;
    unsigned short* const cast = e.cast ? e.cast + c_off : nullptr;
    for (int unit = w; unit < 4 * MT; unit += W) {
        const int i = unit / 4, t = unit % 4;
        float v[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) v[j] = part[unit * NT * 64 + j * 64 + lane];
        for (int o = 1; o < W; ++o)
#pragma unroll
            for (int j = 0; j < NT; ++j) v[j] += part[(o * MT * 4 + unit) * NT * 64 + j * 64 + lane];
        OA orow;  // the rows of the lane that held fragment row 4 (l / 16) + t
        orow.init(p.a, p.a_sm, p.a_sk, m0, p.M, (lane >> 4) * 4 + t);
        if (!orow.owns(i, p.M)) continue;
        const long long at = (long long)orow.mn(i) * p.N;
        if (e.kind == ORMI_GEMM_EPI_NONE) {
            if constexpr (!B_KC && NT == 4) {
                if (ob.owns(0, p.N)) *(f32x4_any*)(c + at + ob.mn(0)) = f32x4_t{v[0], v[1], v[2], v[3]};
                else
#pragma unroll
                    for (int j = 1; j < NT; ++j)
                        if (ob.owns(j, p.N)) c[at + ob.mn(j)] = v[j];
            } else {
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    if (ob.owns(j, p.N)) c[at + ob.mn(j)] = v[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                if (!ob.owns(j, p.N)) continue;
                const int n = ob.mn(j);
                const float dv = epi_reads_d(e) ? e.d[d_off + orow.mn(i) * e.d_sm + n * e.d_sn] : 0.0f;
                epi_store(e, sv, c, aux, cast, at + n, dv, v[j]);
            }
        }
    }
}

template <typename Tr, int MT, int NT>
void launch(const GemmParams& p, dim3 grid, int waves, bool a_kc, bool b_kc) {
    const size_t lds = (size_t)waves * MT * NT * 64 * sizeof(f32x4_t);
    if (a_kc && b_kc) gemm_direct_kernel<Tr, MT, NT, true, true><<<grid, 64 * waves, lds>>>(p);
    else if (a_kc) gemm_direct_kernel<Tr, MT, NT, true, false><<<grid, 64 * waves, lds>>>(p);
    else if (b_kc) gemm_direct_kernel<Tr, MT, NT, false, true><<<grid, 64 * waves, lds>>>(p);
    else gemm_direct_kernel<Tr, MT, NT, false, false><<<grid, 64 * waves, lds>>>(p);
}
template <typename Tr>
void launch_cfg(int mt, int nt, const GemmParams& p, dim3 grid, int waves, bool a_kc, bool b_kc) {
    if (mt == 1 && nt == 2) launch<Tr, 1, 2>(p, grid, waves, a_kc, b_kc);
    else if (mt == 1) launch<Tr, 1, 4>(p, grid, waves, a_kc, b_kc);
    else if (nt == 1) launch<Tr, 4, 1>(p, grid, waves, a_kc, b_kc);
    else if (mt == 2 && nt == 2) launch<Tr, 2, 2>(p, grid, waves, a_kc, b_kc);
    else if (mt == 2) launch<Tr, 2, 4>(p, grid, waves, a_kc, b_kc);
    else launch<Tr, 4, 4>(p, grid, waves, a_kc, b_kc);
}

}  // namespace

// Tile (in 16-element fragments) and waves per work-group for a product, or
// mt = 0 when an mn-contiguous operand has fewer rows (columns) than a fragment
// load takes, up to 4: the other kernels run it.
DirectPlan gemm_direct_plan(const ormi_gemm_desc* d, long long batch, bool a_kc, bool b_kc) {
    DirectPlan r;
    const long long cus = compute_units();
    const bool f32 = d->dtype == ORMI_DTYPE_F32;
    auto tiles = [&](int mt, int nt) {
        return (long long)((d->M + 16 * mt - 1) / (16 * mt)) * ((d->N + 16 * nt - 1) / (16 * nt)) * batch;
    };
    // Up to 16 rows: 64 columns per work-group, a whole cache line of each k-row of
    // 16-bit weights; 32 where the weights are few, for twice the work-groups
    // (bf16 12 x 1000 x 4096 9.4 -> 8.3 us, 6 x 1544 x 2648 12.4 -> 10.3, fp32
    // 16 x 3689 x 640 9.0 -> 6.9; 16 x 5096 x 2656 13.3 -> 13.7, 12 x 4096 x 8192
    // 19.5 -> 24).
    if (d->M <= 16) r.mt = 1, r.nt = (long long)d->N * d->K < (3LL << 22) ? 2 : 4;
    else if (d->N <= 16) r.mt = 4, r.nt = 1;
    else if (tiles(4, 4) >= (f32 ? cus : 2 * cus)) r.mt = 4, r.nt = 4;
    else if (tiles(2, 4) >= 3 * cus / 8) r.mt = 2, r.nt = 4;
    else r.mt = 2, r.nt = 2;
    if ((!a_kc && d->M < r.mt) || (!b_kc && d->N < r.nt)) {
        r.mt = 0;
        return r;
    }
    // Waves: K split until the chip holds six per compute unit (fp32 64 x 64 tiles,
    // whose MFMAs outlast their loads, always four per work-group), each with a
    // few k-steps. Splits across work-groups, summed by the finish pass, only
    // where the tiles leave a quarter of the units idle and a wave still has two
    // k-steps (12 x 8192 by 8192 x 4096 in bf16: 40 us unsplit, 19.8 split by 4),
    // or several if the product is more than a stream of one operand (40 x 4096^2
    // bf16, 16 k-steps a wave: 22 -> 18 us; 1024 x 300 x 1024 fp32, 8: 16 -> 20.6).
    const int kstep = f32 ? 16 : 32;
    const long long t = tiles(r.mt, r.nt), steps = std::max(1, d->K / kstep);
    const int most = std::min(16, 64 / (r.mt * r.nt));
    const long long enough = f32 && r.mt * r.nt == 16 ? 1LL << 40 : 6 * cus;
    while (r.waves < most && t * r.waves < enough && steps >= 4LL * r.waves) r.waves *= 2;
    const long long deep = t < 3 * cus / 8 || r.mt == 1 || r.nt == 1 ? 4 : f32 ? 16 : 8;
    while (r.splits < 8 && t * r.splits < (r.mt == 1 && r.nt == 2 && !f32 ? cus / 2 : 3 * cus / 4) && steps >= deep * r.waves * r.splits) r.splits *= 2;
    if (batch * r.splits > 65535) r.splits = 1;
    return r;
}

void gemm_direct_launch(const ormi_gemm_desc* d, GemmParams& p, long long batch, const DirectPlan& r, bool a_kc, bool b_kc) {
    p.tiles_m = (d->M + 16 * r.mt - 1) / (16 * r.mt);
    p.tiles_n = (d->N + 16 * r.nt - 1) / (16 * r.nt);
    p.splits = r.splits;
    const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, (unsigned)(batch * r.splits));
    if (d->dtype == ORMI_DTYPE_F32) launch_cfg<TrF32>(r.mt, r.nt, p, grid, r.waves, a_kc, b_kc);
    else if (d->dtype == ORMI_DTYPE_BF16) launch_cfg<TrBF16>(r.mt, r.nt, p, grid, r.waves, a_kc, b_kc);
    else launch_cfg<TrF16>(r.mt, r.nt, p, grid, r.waves, a_kc, b_kc);
}
}  // namespace ormi_hip
