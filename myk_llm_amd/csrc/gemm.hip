// Batched bf16 matrix products with fp32 accumulation: the fused head's three products
// (ops/fused_ce.py:70-108) and Muon's batched SYRK and update (ops/muon.py:28-143, 218-268).
//   C[b] = alpha * A[b] B[b] + beta * Add[b]   (bf16 C), or   C[b] = A[b] B[b] + beta * C[b]   (fp32 C)
// with A (M, K) and B (K, N), each stored with either of its dimensions contiguous. SYM: B = A^T,
// only the tiles on and below the diagonal are computed and the others stored as their mirror
// images (the sums run over k in the same order on both sides, so C is exactly symmetric).
//
// Tile. A workgroup owns BM x BN of C: WM x WN waves of MI x NI blocks of 32x32x16 MFMA, n as the
// MFMA row (a lane's registers hold 8 consecutive n in perm32 order) and m as its column. K
// advances 64 per stage through a ring of direct-to-LDS stages. An operand whose K is contiguous is
// staged as rows of 64 and read 16 bytes at a time; one whose M or N is contiguous is staged as 64
// rows of BM / BN and read with the LDS transpose read. Both are swizzled (common.h): 0 bank conflicts.
//
// Pipeline. The barrier of a stage sits before its last k-step: every wave then holds that step's
// operands in registers, so the slot is refilled at once and the next stage's first operands are
// read while the last products run. Half of the waves issue their loads before these products and
// half after them (waves w and w + 4 share a SIMD): a load into LDS holds its wave for about 50
// cycles, and with all waves loading after the barrier the matrix cores idled (8192 x 8192 x 8192:
// 1204 against 1277 TFLOP/s). Loads spread evenly between the products, 32-wide stages in a ring of
// four, four waves of 128 x 128 with the sums in AGPRs and raised wave priority around the products
// all measured slower (1170, 1170, 1085 and 1284 TFLOP/s).
//
// Persistent. A workgroup runs several units and its loads run ahead across their borders, so the
// next unit's first stages land while this one's results are stored (2048 x 65536 x 1024: 327 ->
// 285 us). Results go through 2 KB of LDS per wave so that a store covers whole 128-byte lines
// (452 -> 337 us there); their stores are waited for only when the next unit's own loads are.
//
// Bound by the matrix cores at the clock that the card holds under this load (~1.9 GHz: MFMA busy
// 62 % at 8192 x 8192 x 8192, LDS active 24 %); zeros for data run 35 % faster.
#include "common.h"
#include "gemm_tiles.h"
#include "kernels.h"

namespace mykfa {
namespace {

constexpr int kBK = kGemmBK;
constexpr int kKS = kBK / 16;      // k-steps per stage
constexpr int kCUs = kGemmCUs;
constexpr unsigned kSkip = 0x80000000u;  // an offset outside any buffer: the load returns zero

struct GemmArgs {
    const uint16_t* a;
    const uint16_t* b;
    int64_t a_bs, a_rs, b_bs, b_rs;  // batch and row strides, elements
    int m, n, k;
    void* c;
    const uint16_t* add;
    int64_t c_bs, c_rs, d_bs, d_rs;
    float alpha, beta;
    bool c_vec, d_vec;  // 16-byte rows of C / Add (else 8-byte / 2-byte accesses; SYM only)
    int batch;
    GemmGrid g;
    int per_xcd, units;  // of this launch
};

enum Out { OUT_BF16, OUT_ADD, OUT_F32, OUT_PART, OUT_SYM };  // OUT_BF16: no addend

// One operand's tile of R rows of M or N: R x 64 (K contiguous), or 64 x R (TR: R contiguous).
template <int R, bool TR, int NW>
struct Operand {
    static constexpr int W = TR ? R : kBK;  // contiguous elements per staged row
    static constexpr int CPR = W / 8;       // 16-byte chunks per staged row
    static constexpr int LOADS = R * kBK / 8 / 64 / NW;
    static_assert(R * kBK / 8 % (64 * NW) == 0, "whole loads per wave");
    unsigned voff[LOADS];  // of this wave's loads, the same for every tile
    int64_t rs;
    uint64_t base;
    GemmPart part;

    __device__ inline void offsets(int64_t rstride, int wave, int lane) {
        rs = rstride;
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const int c = (wave * LOADS + j) * 64 + lane;
            const int row = c / CPR, phys = c % CPR;
            voff[j] = (unsigned)(row * (int)(rs * 2) + ((phys ^ lds_swz<W>(row)) << 4));
        }
    }
    // The tile whose first row (column) of `mn` is r0.
    __device__ inline void enter(const uint16_t* p, int mn, int k, int r0) {
        part = gemm_part<TR>(mn, k, r0, R);
        base = reinterpret_cast<uint64_t>(p + (int64_t)part.row0 * rs + part.col0);
    }
    struct Stage {
        i32x4 rsrc;
        int left;  // columns of K from it on
    };
    Stage next;
    __device__ inline Stage stage(int kt) const {
        const GemmSpan s = gemm_span<TR>(part, (int)rs, kt);
        return Stage{buffer_rsrc32(base + ((uint64_t)(unsigned)s.row * (uint64_t)rs + (unsigned)s.col) * 2, s.bytes),
                     part.cols - s.col};
    }
    // This wave's loads of a stage into the tile at LDS address lds. Rows past the matrix read
    // zero through the descriptor; chunks past K through their offset.
    __device__ inline void issue(const Stage& s, uint32_t lds, int wave, int lane) const {
        const i32x4 rsrc = s.rsrc;
        if constexpr (!TR) {
            const int left = s.left;
            if (left < kBK) {
#pragma unroll
                for (int j = 0; j < LOADS; ++j) {
                    const int c = (wave * LOADS + j) * 64 + lane;
                    const int row = c / CPR, logical = (c % CPR) ^ lds_swz<W>(row);
                    dma16(rsrc, lds + (uint32_t)((wave * LOADS + j) * 1024), logical * 8 < left ? voff[j] : kSkip);
                }
                return;
            }
        }
#pragma unroll
        for (int j = 0; j < LOADS; ++j) dma16(rsrc, lds + (uint32_t)((wave * LOADS + j) * 1024), voff[j]);
    }
    // MFMA operand of the 32 rows at rb (in perm32 order with PERM), k-step kk.
    template <bool PERM>
    __device__ static inline s16x8 read(const uint16_t* tile, int rb, int kk, int lane) {
        const int l32 = lane & 31, g = lane >> 5;
        if constexpr (TR) {
            const int G = lane >> 4, jj = lane & 15;
            const int x = PERM ? ((jj & 1) << 1) | ((jj >> 1) & 1) : jj & 3;
            const int col = rb + 16 * (G & 1) + 4 * x;
            const int row = 16 * kk + 8 * (G >> 1) + (jj >> 2);
            return cat4(ds_read_tr(tile + lds_off<W>(row, col)), ds_read_tr(tile + lds_off<W>(row + 4, col)));
        } else {
            const int row = rb + (PERM ? perm32(l32) : l32);
            return *reinterpret_cast<const s16x8*>(tile + row * W + (((2 * kk + g) ^ lds_swz<W>(row)) << 3));
        }
    }
};

// 8 elements of a row of which `left` exist.
__device__ inline void store8(uint16_t* c, s16x8 w, int left, bool vec) {
    if (left >= 8) {
        if (vec) {
            st16(c, w);
        } else {
            *reinterpret_cast<s16x4*>(c) = s16x4{w[0], w[1], w[2], w[3]};
            *reinterpret_cast<s16x4*>(c + 4) = s16x4{w[4], w[5], w[6], w[7]};
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (e < left) c[e] = (uint16_t)w[e];
    }
}
// The first `left` of 8 elements, zeros after them.
__device__ inline s16x8 first8(s16x8 w, int left) {
#pragma unroll
    for (int e = 0; e < 8; ++e) w[e] = e < left ? w[e] : (short)0;
    return w;
}
__device__ inline s16x8 load8(const uint16_t* d, int left, bool vec) {
    if (vec && left >= 8) return ld16(d);
    s16x8 w = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (e < left) w[e] = (short)d[e];
    return w;
}

template <int WM, int WN, int MI, int NI, int STAGES, int OCC, bool AT, bool BT, int OUT>
__global__ __launch_bounds__(WM * WN * 64, OCC) void gemm_kernel(GemmArgs p) {
    constexpr int NW = WM * WN, BM = WM * MI * 32, BN = WN * NI * 32;
    static_assert(NI % 2 == 0, "results are stored 64 columns at a time");
    using OpA = Operand<BM, AT, NW>;
    using OpB = Operand<BN, BT, NW>;
    constexpr int LOADS = OpA::LOADS + OpB::LOADS;
    constexpr int SLOT = (BM + BN) * kBK;
    constexpr int STORES = MI * NI / 2 * 4;  // 16-byte stores per wave of a full bf16 tile
    __shared__ __attribute__((aligned(16))) uint16_t smem[STAGES * SLOT + NW * 1024];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, g = lane >> 5;
    const int wm = wave % WM, wn = wave / WM;

    // The dispatcher deals workgroup i to XCD i % 8: XCD x takes one contiguous run of the unit
    // list, its workgroups unit `first`, then every step-th.
    const int xcd = (int)(blockIdx.x % kXcds), step = (int)(gridDim.x / kXcds);
    const int end = min((xcd + 1) * p.per_xcd, p.units);
    const int first = xcd * p.per_xcd + (int)(blockIdx.x / kXcds);
    if (first >= end) return;
    // Unit -> (batch, split, tile); SYM: row by row of the lower triangle.
    auto tile_of = [&](int unit) {
        if constexpr (OUT == OUT_SYM) {
            const int tiles = p.g.tm * (p.g.tm + 1) / 2, x = unit % tiles, bidx = unit / tiles;
            int r = (int)((sqrtf(8.0f * (float)x + 1.0f) - 1.0f) * 0.5f);
            while (r * (r + 1) / 2 > x) --r;
            while ((r + 1) * (r + 2) / 2 <= x) ++r;
            r = __builtin_amdgcn_readfirstlane(r);
            return GemmTile{bidx, bidx, r * BM, (x - r * (r + 1) / 2) * BN, 0, p.g.stages};
        } else {
            return gemm_tile(p.g, p.k, unit, BM, BN);
        }
    };

    // The loads run ahead of the products: stage lk of unit lu (tile lt) goes to slot lslot next;
    // `ahead` stages are loaded and not yet consumed.
    OpA oa;
    OpB ob;
    oa.offsets(p.a_rs, wave, lane);
    ob.offsets(p.b_rs, wave, lane);
    int lu = first, lk = 0, lslot = 0, ahead = 0;
    GemmTile lt = tile_of(lu);
    auto enter = [&]() {
        oa.enter(p.a + lt.bidx * p.a_bs, p.m, p.k, lt.m0);
        ob.enter(p.b + lt.bidx * p.b_bs, p.n, p.k, lt.n0);
    };
    enter();
    const uint32_t lds0 = lds_addr(&smem[0]);
    // The symmetric products and the smallest tiles compute the next stage's descriptors before they wait for
    // the one before: with a CU to themselves, the time from a stage's landing to the next one's loads is their
    // chain (symmetric 9 x 1024 x 4096 60.3 -> 59.0 us, 9 x 512 x 2048 21.1 -> 19.6, 1 x 1024 x 4096 34.6 -> 32.5).
    // The 256 x 256 tiles lose by it (8192 x 1024 x 65536 922 -> 942: more scalar registers spilled).
    constexpr bool kAhead = OUT == OUT_SYM || NW == 2;
    auto prepare = [&]() {
        oa.next = oa.stage(lt.kt0 + lk);
        ob.next = ob.stage(lt.kt0 + lk);
    };
    auto issue = [&]() {
        if (lu >= end) return;
        const uint32_t at = lds0 + (uint32_t)(lslot * SLOT * 2);
        oa.issue(kAhead ? oa.next : oa.stage(lt.kt0 + lk), at, wave, lane);
        ob.issue(kAhead ? ob.next : ob.stage(lt.kt0 + lk), at + BM * kBK * 2, wave, lane);
        ++ahead;
        lslot = lslot + 1 == STAGES ? 0 : lslot + 1;
        if (++lk == lt.nk) {
            lk = 0;
            lu += step;
            if (lu < end) {
                lt = tile_of(lu);
                enter();
            }
        }
    };
#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
        if (kAhead) prepare();
        issue();
    }

    f32x16 acc[MI][NI];
    s16x8 av[2][MI], bv[2][NI];
    int slot = 0;  // of the stage being consumed
    auto read = [&](int kk, int buf) {
        const uint16_t* ta = &smem[slot * SLOT];
        const uint16_t* tb = ta + BM * kBK;
#pragma unroll
        for (int j = 0; j < NI; ++j) bv[buf][j] = OpB::template read<true>(tb, (wn * NI + j) * 32, kk, lane);
#pragma unroll
        for (int i = 0; i < MI; ++i) av[buf][i] = OpA::template read<false>(ta, (wm * MI + i) * 32, kk, lane);
    };
    auto multiply = [&](int buf) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j) acc[i][j] = BF16::mfma32(bv[buf][j], av[buf][i], acc[i][j]);
    };
    // The oldest stage not consumed has landed for every wave: each waits for its own loads, then
    // the barrier. While pend > 0 that stage was issued before a full tile's STORES stores.
    int pend = 0;
    auto landed = [&]() {
        asm volatile("" ::: "memory");
        if (pend > 0 && ahead == STAGES - 1) wait_vmcnt<(STAGES - 2) * LOADS + STORES>();
        else ring_wait<LOADS, STAGES>(ahead - 1);
        --pend;
        barrier_lds();
        asm volatile("" ::: "memory");
    };
    asm volatile("" ::: "memory");
    if (ahead == STAGES) wait_vmcnt<(STAGES - 1) * LOADS>();
    else wait_vmcnt<0>();
    barrier_lds();
    asm volatile("" ::: "memory");
    read(0, 0);

    for (int unit = first; unit < end; unit += step) {
        const GemmTile t = tile_of(unit);
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
        for (int kt = 0; kt < t.nk; ++kt) {
#pragma unroll
            for (int kk = 0; kk < kKS - 1; ++kk) {
                read(kk + 1, (kk + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
                multiply(kk & 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            --ahead;
            slot = slot + 1 == STAGES ? 0 : slot + 1;
            const bool more = ahead > 0;
            if (more) {
                if (kAhead) prepare();
                landed();
                if (NW < 8 || wave < NW / 2) issue();
                read(0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            multiply((kKS - 1) & 1);
            __builtin_amdgcn_sched_barrier(0);
            if (NW == 8 && more && wave >= NW / 2) {
                issue();
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // Register r of lane (g, l32) of block (i, j) is C at n = 32 j + out_row32(r, g), m = 32 i + l32.
        uint16_t* tr = &smem[STAGES * SLOT] + wave * 1024;
        const bool full = t.m0 + BM <= p.m && t.n0 + BN <= p.n;
        if constexpr (OUT == OUT_BF16 || OUT == OUT_ADD || OUT == OUT_SYM) {
            const uint16_t* add = p.add ? p.add + t.bidx * p.d_bs : nullptr;
            uint16_t* cb = static_cast<uint16_t*>(p.c) + t.bidx * p.c_bs;
            pend = full && OUT == OUT_BF16 ? STAGES - 1 : 0;
            // Columns stored: OUT_BF16 and OUT_ADD fill a row's pad up to a multiple of 8 with zeros, whatever the
            // operands hold there (an infinity in A's row times the zeros past B's last row is a NaN); OUT_SYM
            // stores none.
            const int n_end = OUT == OUT_SYM ? p.n : (p.n + 7) & ~7;
#pragma unroll
            for (int i = 0; i < MI; ++i)
#pragma unroll
                for (int jp = 0; jp < NI; jp += 2) {
                    const int mb = t.m0 + (wm * MI + i) * 32, nb = t.n0 + (wn * NI + jp) * 32;
                    s16x8 w[2][2];
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            float v[8];
#pragma unroll
                            for (int e = 0; e < 8; ++e) v[e] = acc[i][jp + j][8 * h + e] * p.alpha;
                            if (OUT != OUT_BF16 && add) {
                                const int m = mb + l32, n = nb + 32 * j + 16 * h + 8 * g;
                                if (m < p.m && n < p.n) {
                                    const s16x8 x = load8(add + (int64_t)m * p.d_rs + n, n_end - n, OUT == OUT_ADD || p.d_vec);
#pragma unroll
                                    for (int e = 0; e < 8; ++e) v[e] += p.beta * BF16::to_float((uint16_t)x[e]);
                                }
                            }
                            const u32x4 u = {BF16::pack2(v[0], v[1]), BF16::pack2(v[2], v[3]), BF16::pack2(v[4], v[5]),
                                             BF16::pack2(v[6], v[7])};
                            w[j][h] = __builtin_bit_cast(s16x8, u);
                        }
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        // 16 rows x 64 columns at a time, 16-byte chunk c of row r at c ^ (r mod 8).
                        if (q % 2 == 0) {
                            wave_fence();
                            if (l32 / 16 == q / 2) {
#pragma unroll
                                for (int j = 0; j < 2; ++j)
#pragma unroll
                                    for (int h = 0; h < 2; ++h)
                                        st16(tr + l32 % 16 * 64 + (((4 * j + 2 * h + g) ^ (l32 & 7)) << 3), w[j][h]);
                            }
                            wave_fence();
                        }
                        const int r = 8 * q + (lane >> 3), ch = lane & 7, m = mb + r, n = nb + 8 * ch;
                        s16x8 y = *reinterpret_cast<const s16x8*>(tr + r % 16 * 64 + ((ch ^ (r & 7)) << 3));
                        if (full || (m < p.m && n < n_end)) {
                            uint16_t* c = cb + (int64_t)m * p.c_rs + n;
                            if constexpr (OUT == OUT_SYM) {
                                store8(c, y, n_end - n, p.c_vec);
                            } else {
                                if (!full) y = first8(y, p.n - n);
                                st16(c, y);
                            }
                        }
                    }
                    if (OUT == OUT_SYM && t.m0 != t.n0) {
                        // The mirror image: 32 columns x 32 rows at a time.
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            wave_fence();
#pragma unroll
                            for (int h = 0; h < 2; ++h)
#pragma unroll
                                for (int e = 0; e < 8; ++e) tr[(16 * h + 8 * g + e) * 32 + l32] = (uint16_t)w[j][h][e];
                            wave_fence();
#pragma unroll
                            for (int q = 0; q < 2; ++q) {
                                const int r = 16 * q + (lane >> 2), ch = lane & 3, n = nb + 32 * j + r, m = mb + 8 * ch;
                                const s16x8 y = *reinterpret_cast<const s16x8*>(tr + r * 32 + 8 * ch);
                                if (n < p.n && m < p.m) store8(cb + (int64_t)n * p.c_rs + m, y, p.m - m, p.c_vec);
                            }
                        }
                    }
                }
        } else {
            pend = 0;
            float* trf = reinterpret_cast<float*>(tr);
            float* cb = static_cast<float*>(p.c) + (OUT == OUT_PART ? (int64_t)t.outer * p.m * p.c_rs : t.bidx * p.c_bs);
            const bool add = OUT == OUT_F32 && p.beta != 0.f;
            const int n_end = (p.n + 7) & ~7;
            // Block x = i NI + j: 32 x 32. The sums that a block adds to are loaded before its exchange
            // (loading the next block's as well costs 35 spilled registers: 494 against 346 us at
            // 65536 x 1024 x 2048).
            auto at = [&](int x, int q) {
                const int m = t.m0 + (wm * MI + x / NI) * 32 + 8 * q + (lane >> 3);
                const int n = t.n0 + (wn * NI + x % NI) * 32 + 4 * (lane & 7);
                return m < p.m && n < n_end ? cb + (int64_t)m * p.c_rs + n : nullptr;
            };
#pragma unroll
            for (int x = 0; x < MI * NI; ++x) {
                f32x4 old[4];
                if (add) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float* c = at(x, q);
                        if (c) old[q] = *reinterpret_cast<const f32x4*>(c);
                    }
                }
                const f32x16& v = acc[x / NI][x % NI];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // 16 rows at a time, 16-byte chunk c of row r at c ^ (r mod 8).
                    if (q % 2 == 0) {
                        wave_fence();
                        if (l32 / 16 == q / 2) {
#pragma unroll
                            for (int u = 0; u < 4; ++u) {
                                const int ch = 4 * (u >> 1) + 2 * g + (u & 1);
                                *reinterpret_cast<f32x4*>(trf + l32 % 16 * 32 + ((ch ^ (l32 & 7)) << 2)) =
                                    f32x4{v[4 * u], v[4 * u + 1], v[4 * u + 2], v[4 * u + 3]};
                            }
                        }
                        wave_fence();
                    }
                    const int r = 8 * q + (lane >> 3), ch = lane & 7;
                    f32x4 w = *reinterpret_cast<const f32x4*>(trf + r % 16 * 32 + ((ch ^ (r & 7)) << 2));
                    if (add) w += old[q] * p.beta;
                    float* c = at(x, q);
                    // Past the caches, whose panels the sums would evict (285 -> 260 us for 268 MB written
                    // once); bf16 results are the next launch's input and stay (the fused head 7837 against
                    // 7599 us with them past the caches).
                    if (c) __builtin_nontemporal_store(w, reinterpret_cast<f32x4*>(c));
                }
            }
        }
    }
}

// The K splits' fp32 products, summed in order and rounded: 8 columns a lane, zeros past n.
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float* part, int splits, int64_t stride, uint16_t* c,
                                                          int64_t c_bs, int64_t c_rs, int batch, int m, int n,
                                                          float alpha) {
    const int n8 = (n + 7) / 8;
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t per = (int64_t)m * n8;
    if (idx >= per * batch) return;
    const int64_t b = idx / per, r = idx % per / n8, col = idx % n8 * 8;
    const float* s = part + b * splits * stride + (r * n8) * 8 + col;
    f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;
    for (int i = 0; i < splits; ++i, s += stride) {
        lo += *reinterpret_cast<const f32x4*>(s);
        hi += *reinterpret_cast<const f32x4*>(s + 4);
    }
    lo *= alpha;
    hi *= alpha;
    const u32x4 w = {BF16::pack2(lo[0], lo[1]), BF16::pack2(lo[2], lo[3]), BF16::pack2(hi[0], hi[1]),
                     BF16::pack2(hi[2], hi[3])};
    st16(c + b * c_bs + r * c_rs + col, first8(__builtin_bit_cast(s16x8, w), n - (int)col));
}

template <int WM, int WN, int MI, int NI, int STAGES, int OCC, bool AT, bool BT, int OUT>
hipError_t launch(GemmArgs a, hipStream_t s) {
    constexpr int LDS = (STAGES * (WM * MI + WN * NI) * 32 * kBK + WM * WN * 1024) * 2;
    constexpr int PER_XCD = kCUs / kXcds * (LDS > 80 * 1024 ? 1 : 2);  // resident workgroups
    a.per_xcd = (a.units + kXcds - 1) / kXcds;
    const int per = a.per_xcd < PER_XCD ? a.per_xcd : PER_XCD;
    hipLaunchKernelGGL((gemm_kernel<WM, WN, MI, NI, STAGES, OCC, AT, BT, OUT>), dim3(per * kXcds), dim3(WM * WN * 64), 0, s,
                       a);
    return hipGetLastError();
}

// Tiles, largest first: 256 x 256 in 8 waves (2 stages, one workgroup per CU), 128 x 128 in 4 (2
// stages, two per CU), 64 x 64 in 2 (4 stages, two per CU).
enum Size { BIG, MID, SMALL };
long long tile_count(int m, int n, int batch, int t) {
    return (long long)((m + t - 1) / t) * ((n + t - 1) / t) * batch;
}

template <bool AT, bool BT, int OUT>
hipError_t launch_size(GemmArgs a, Size size, hipStream_t s) {
    const int side = 256 >> size;
    a.g.tm = (a.m + side - 1) / side;
    a.g.tn = (a.n + side - 1) / side;
    a.g.stages = (gemm_stages(a.k) + a.g.splits - 1) / a.g.splits;
    const long long units =
        (OUT == OUT_SYM ? (long long)a.g.tm * (a.g.tm + 1) / 2 : (long long)a.g.tm * a.g.tn) * a.batch * a.g.splits;
    if (units > (1ll << 30)) return hipErrorInvalidValue;
    a.units = (int)units;
    if (size == SMALL) return launch<2, 1, 1, 2, 4, 1, AT, BT, OUT>(a, s);
    if (size == MID) return launch<2, 2, 2, 2, 2, 2, AT, BT, OUT>(a, s);
    // A last round of at most half the CUs runs as quarters, two of which a CU holds: nine products
    // of 1024 x 4096 x 1024 (576 units) 103 -> 95 us.
    const int rest = a.units % kCUs;
    if (OUT != OUT_SYM && a.units > kCUs && rest > 0 && rest <= kCUs / 2) {
        a.units -= rest;
        const hipError_t e = launch<2, 4, 4, 2, 2, 2, AT, BT, OUT>(a, s);
        if (e != hipSuccess) return e;
        a.g.first_unit = a.units;
        a.g.quarters = true;
        a.units = 4 * rest;
        return launch<2, 2, 2, 2, 2, 2, AT, BT, OUT>(a, s);
    }
    return launch<2, 4, 4, 2, 2, 2, AT, BT, OUT>(a, s);
}

// The largest tile whose units come to at least 3/4 of the CUs: fewer leave more of the chip idle
// than the smaller tile costs in operand traffic.
struct Plan {
    Size size;
    int splits;
};
// Stages of the product that one more part of every result costs in fp32 partials written and read
// back (256 x 256 x 8 bytes at the copy rate against 1.6 us a stage, both over the whole chip).
constexpr double kPartStages = 19;

// Rounds of the CUs that `units` of the 256 x 256 tiles take; a short last round runs as quarters.
double big_rounds(long long units) {
    const long long rest = units % kCUs;
    return (double)(units / kCUs) + (rest == 0 ? 0. : units > kCUs && rest <= kCUs / 2 ? .85 : 1.);
}
// Parts of K for the 256 x 256 tiles that take the least time, over up to three rounds. With one
// round only, tiles just above a half or a third of the CUs went to the 128 x 128 tile whole: rows x
// 1024 x 65536 with 10000 rows (160 tiles, now in 3 parts) 1996 -> 1260 us, 5632 (88, 8) 957 -> 728, 6144
// (96, 8) 869 -> 811; counts that divide the CUs evenly as they were.
int big_splits(long long tiles, int stages) {
    int best = 1;
    double least = 0;
    for (int s = 1; s == 1 || (s <= stages / 16 && tiles * s <= 3 * kCUs); ++s) {
        const int per = (stages + s - 1) / s;
        if (s > 1 && (stages + per - 1) / per != s) continue;  // every split holds a stage
        const double cost = big_rounds(tiles * s) * kCUs * per / tiles + (s > 1 ? kPartStages * s : 0);
        if (s == 1 || cost < least) {
            best = s;
            least = cost;
        }
    }
    return best;
}
// K is split only for bf16 results without an addend, into at least 16 stages each.
Plan plan_of(const mykfa_gemm_params& p) {
    const int stages = (p.k + kBK - 1) / kBK;
    const bool can_split = p.c_dtype == MYKFA_BF16 && p.add == nullptr;
    for (int size = BIG; size <= SMALL; ++size) {
        const long long tiles = tile_count(p.m, p.n, p.batch, 256 >> size);
        int splits = 1;
        if (can_split && size == BIG) {
            splits = big_splits(tiles, stages);
        } else if (can_split && tiles <= kCUs / 2) {
            splits = (int)(kCUs / tiles);
            if (splits > stages / 16) splits = stages / 16;
            if (splits < 1) splits = 1;
            const int per = (stages + splits - 1) / splits;
            splits = stages > 0 ? (stages + per - 1) / per : 1;  // every split holds a stage
        }
        if (size == SMALL || tiles * splits >= kCUs * 3 / 4) return Plan{(Size)size, splits};
    }
    return Plan{SMALL, 1};
}

}  // namespace

size_t gemm_workspace_bytes(const mykfa_gemm_params& p) {
    if (p.batch <= 0 || p.m <= 0 || p.n <= 0 || p.symmetric) return 0;
    const Plan plan = plan_of(p);
    return plan.splits > 1 ? (size_t)plan.splits * p.batch * p.m * ((p.n + 7) & ~7) * sizeof(float) : 0;
}

hipError_t launch_gemm(const mykfa_gemm_params& p, void* ws, hipStream_t stream) {
    GemmArgs a{};
    a.a = static_cast<const uint16_t*>(p.a);
    a.b = static_cast<const uint16_t*>(p.b);
    a.a_bs = p.a_batch_stride; a.a_rs = p.a_row_stride;
    a.b_bs = p.b_batch_stride; a.b_rs = p.b_row_stride;
    a.m = p.m; a.n = p.n; a.k = p.k; a.batch = p.batch;
    a.c = p.c;
    a.c_bs = p.c_batch_stride; a.c_rs = p.c_row_stride;
    a.add = static_cast<const uint16_t*>(p.add);
    a.d_bs = p.add_batch_stride; a.d_rs = p.add_row_stride;
    a.alpha = p.alpha; a.beta = p.beta;
    if (p.symmetric) {
        a.b = a.a;
        a.b_bs = a.a_bs; a.b_rs = a.a_rs;
        const auto vec = [](const void* ptr, int64_t bs, int64_t rs) {
            return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0 && (bs & 7) == 0 && (rs & 7) == 0;
        };
        a.c_vec = vec(p.c, a.c_bs, a.c_rs);
        a.d_vec = vec(p.add, a.d_bs, a.d_rs);
        a.g.splits = 1;
        const long long t = (p.m + 127) / 128;
        return launch_size<false, false, OUT_SYM>(a, p.batch * (t * (t + 1) / 2) >= kCUs * 3 / 4 ? MID : SMALL, stream);
    }
    a.c_vec = a.d_vec = true;
    const Plan plan = plan_of(p);
    a.g.splits = plan.splits;
    if (p.c_dtype == MYKFA_FP32) return launch_size<true, true, OUT_F32>(a, plan.size, stream);
    if (plan.splits > 1) {
        const int n8 = (p.n + 7) / 8;
        a.c = ws;
        a.c_rs = (int64_t)n8 * 8;
        const hipError_t e = p.b_transposed ? launch_size<false, false, OUT_PART>(a, plan.size, stream)
                                            : launch_size<false, true, OUT_PART>(a, plan.size, stream);
        if (e != hipSuccess) return e;
        const int64_t lanes = (int64_t)p.batch * p.m * n8;
        hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, stream,
                           static_cast<const float*>(ws), plan.splits, (int64_t)p.m * n8 * 8,
                           static_cast<uint16_t*>(p.c), p.c_batch_stride, p.c_row_stride, p.batch, p.m, p.n, p.alpha);
        return hipGetLastError();
    }
    if (p.add)
        return p.b_transposed ? launch_size<false, false, OUT_ADD>(a, plan.size, stream)
                              : launch_size<false, true, OUT_ADD>(a, plan.size, stream);
    return p.b_transposed ? launch_size<false, false, OUT_BF16>(a, plan.size, stream)
                          : launch_size<false, true, OUT_BF16>(a, plan.size, stream);
}

hipError_t launch_syrk(const mykfa_syrk_params& p, hipStream_t stream) {
    mykfa_gemm_params g{};
    g.a = p.x;
    g.a_batch_stride = p.x_batch_stride; g.a_row_stride = p.x_row_stride;
    g.c = p.out;
    g.c_batch_stride = p.out_batch_stride; g.c_row_stride = p.out_row_stride;
    g.add = p.bias;
    g.add_batch_stride = p.bias_batch_stride; g.add_row_stride = p.bias_row_stride;
    g.batch = p.batch; g.m = g.n = p.m; g.k = p.k;
    g.symmetric = 1;
    g.alpha = p.alpha; g.beta = p.beta;
    g.c_dtype = MYKFA_BF16;
    return launch_gemm(g, nullptr, stream);
}

}  // namespace mykfa
