// Attention at head dims up to 64 (padded width 64): dense, and the PISA list
// of selected blocks and centroids with the merge and first-order correction;
// and small dense calls at head dims up to 128, which read K and V in place
// (attention.hip describes the computation; the operand tables, the transposed
// scores and the lazy softmax are the same; it also runs the dense packed calls
// that give each SIMD at most one wave, dense_d64_one_wave).
#include "attention_softmax.hpp"
#include "kernels.hpp"

namespace pisa {

namespace {

constexpr int NT = 2;  // 32-row query tiles of a 64-row block
constexpr int kRawFlags = 0x00020000;  // untyped 32-bit buffer data format

// Width 64 runs two waves per SIMD (256 registers each).  What bounds the loop, from
// register-only loops of its instruction mix (one MI355X, random operands):
// per 32-key half chunk the 16 MFMAs hold the matrix core 512 cycles and the
// vector issue port about 15 cycles each, the 94 ordinary softmax instructions
// 3.9 and the 32 exponentials 8 each, 863 cycles in all (measured 858 with two
// waves, 889 with one), and each 1 KB operand fragment loaded adds about 10
// cycles with two waves per SIMD and 22 with one: 490 ns per half chunk with
// all operands from L2, at the 1.84-2.0 GHz that power leaves (fewer vector
// instructions lower the cycles and the clock together).  The kernel takes
// 540-580 ns; the one-wave kernel before it 555-610.  256 registers hold one
// set of key and one of value fragments, each reloaded for the next half chunk
// as soon as its products are issued: the other wave covers the latency.
//
// W waves share one query block, each walking a contiguous part of its chunk
// list for all 64 query rows, and merge through LDS (fixed order, so the
// result is reproducible): per column the running maxima, then the parts of O
// scaled to the common maximum and summed by output units.  Every key and value
// byte is still loaded once per query block.  launch_t chooses W.
//
// DIRECT (small dense calls): K and V are read from the caller's rows instead of
// the packed tables, so no packing launch runs before.  The key operand is 16
// bytes of one row per lane; of the values a lane reads MD consecutive dims of
// every key row it contracts (as in fixed_block_mfma_kernel), so output tile md
// holds dims MD i + md of accumulator row i.  Each chunk costs more loads (at
// width 64 20 instead of 8 per half: 4 of keys, from 32 rows each, and 16 of
// values, from two rows each): dense_rows_in_place says when that is the better
// trade.  Width 128 exists in this form only (340 registers, one wave per SIMD).
template <typename T, int D, bool SPARSE, bool TAIL, int W, bool DIRECT>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(D <= 64 ? 2 : 1, D <= 64 ? 2 : 1)))
void attention_parts_kernel(AttnArgs a, KvRows kv, const int32_t* __restrict__ sel,
                            const uint32_t* __restrict__ selmask) {
    static_assert(!DIRECT || (!SPARSE && !TAIL), "rows are read in place by the dense kernel only");
    static_assert(D == 64 || (D == 128 && DIRECT), "packed tables of other widths: attention.hip");
    constexpr int KT = D / 16;  // 16-deep k-steps of the score products
    constexpr int MD = D / 32;  // 32-dim output tiles
    constexpr int kBlockBytes = D * kBlock * 2;
    typedef typename Elem<T>::vec8 vec8;
    const int lane = threadIdx.x & 63;
    const int wave = W > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
    const int half = lane >> 5;
    const int col = lane & 31;
    const float c = a.scale_log2;
    const int work = xcd_remap(blockIdx.x, gridDim.x);
    const int bh = work / a.q_blocks;
    const int qb = work - bh * a.q_blocks;

    // ---- query rows: qreg[nt][t] = Q[row 32nt + col][16t + 8half .. +7], zero past the real head dim
    vec8 qreg[NT][KT];
    const int qbase = a.qmap.block_base(qb);
    int q_off[NT];
    {
        const char* q_head = a.q.data + a.q.row(bh, 0) * (int64_t)sizeof(T) + half * 16;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            q_off[nt] = a.qmap.intra_offset(32 * nt + col);
            const int tok = min(qbase + q_off[nt], a.q_tokens - 1);  // rows past the end are never stored
            const char* p = q_head + (int64_t)tok * a.q.st * (int64_t)sizeof(T);
#pragma unroll
            for (int t = 0; t < KT; ++t) {
                if (t * 16 + half * 8 < a.head_dim) {
                    qreg[nt][t] = load8<vec8>(p + t * 32);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) qreg[nt][t][e] = T(0.0f);
                }
            }
        }
    }

    f32x16 o[MD][NT];
#pragma unroll
    for (int md = 0; md < MD; ++md)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int v = 0; v < 16; ++v) o[md][nt][v] = 0.0f;
    float nm[NT], mth[NT], l[NT], lt[NT];  // running max as -m and m + kLazyRescale (rescale_to)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        nm[nt] = 0.0f;
        mth[nt] = -__builtin_inff();
        l[nt] = 0.0f;
        lt[nt] = 0.0f;
    }

    // ---- chunk list: [0, n_exact) exact blocks, [n_exact, n_chunks) centroid
    // chunks; this wave's part is [lo, hi), never empty (W <= n_chunks)
    const int n_exact = SPARSE ? a.exact : a.kv_blocks;
    const int n_chunks = n_exact + (TAIL ? a.npad / kBlock : 0);
    const int lo = wave * n_chunks / W;
    const int hi = (wave + 1) * n_chunks / W;
    const int32_t* my_idx = SPARSE ? sel + ((int64_t)bh * a.q_blocks + qb) * a.exact : nullptr;
    const uint32_t* my_mask = TAIL ? selmask + ((int64_t)bh * a.q_blocks + qb) * a.mask_words : nullptr;
    // Packed tables of this head as buffer resources (reads past a table return
    // zero).  Exact or centroid chunk is a choice between base pointers and
    // sizes, which stay in scalar registers; a choice between resources would go
    // through private memory, with a wait for every load in flight.
    const int tab_bytes = a.kv_blocks * kBlockBytes;
    const int cen_bytes = TAIL ? a.npad * D * 2 : 0;
    const char* const kp = a.kp + (int64_t)bh * tab_bytes;
    const char* const vp = a.vp + (int64_t)bh * tab_bytes;
    const char* const kc = TAIL ? a.kbar + (int64_t)bh * cen_bytes : kp;
    const char* const vc = TAIL ? a.vbar_t + (int64_t)bh * cen_bytes : vp;
    auto table = [&](bool tail, const char* exact, const char* centroids) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)(TAIL && tail ? centroids : exact), (short)0,
                                                 TAIL && tail ? cen_bytes : tab_bytes, kRawFlags);
    };
    const int lane_off = lane * 16;

    // DIRECT: the rows of this head.  The whole byte offset of a load is its
    // vector offset, which the hardware checks against the size, so what lies
    // past the last row (or past its last dim) reads as zero.
    const int k_row = DIRECT ? (int)kv.k.st * 2 : 0, v_row = DIRECT ? (int)kv.v.st * 2 : 0;  // bytes
    const __amdgpu_buffer_rsrc_t kr_rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(DIRECT ? kv.k.data + kv.k.row(bh, 0) * 2 : a.kp), (short)0,
        DIRECT ? (a.kv_tokens - 1) * k_row + a.head_dim * 2 : 0, kRawFlags);
    const __amdgpu_buffer_rsrc_t vr_rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(DIRECT ? kv.v.data + kv.v.row(bh, 0) * 2 : a.vp), (short)0,
        DIRECT ? (a.kv_tokens - 1) * v_row + a.head_dim * 2 : 0, kRawFlags);
    const bool all_dims = a.head_dim >= D;

    auto is_tail = [&](int x) { return TAIL && min(x, n_chunks - 1) >= n_exact; };
    auto table_row = [&](int x) -> int {  // block id, or centroid chunk id; past the list, its last chunk again
        x = min(x, n_chunks - 1);
        if (TAIL && x >= n_exact) return x - n_exact;
        return SPARSE ? my_idx[x] : x;
    };
    auto ld_frag = [&](__amdgpu_buffer_rsrc_t rs, int off, int frag) -> vec8 {
        const int soff = __builtin_amdgcn_readfirstlane(off + (frag >> 2) * 4096);
        return __builtin_bit_cast(vec8,
                                  __builtin_amdgcn_raw_buffer_load_b128(rs, lane_off + (frag & 3) * 1024, soff, 0));
    };

    vec8 kf[KT];     // key fragments of the half chunk scored next
    vec8 vf[DIRECT ? 1 : MD][2];  // value fragments of the half chunk multiplied next
    // DIRECT: dims MD col .. + MD - 1 of its keys 16ss + 8(e/4) + 4half + e%4, two to a word
    uint32_t vr[DIRECT ? 2 : 1][8][MD / 2];
    auto load_k = [&](bool tail, int row, int mt) {
        if constexpr (DIRECT) {
            const int off = (row * kBlock + mt * 32 + col) * k_row + half * 16;
#pragma unroll
            for (int t = 0; t < KT; ++t)
                kf[t] = __builtin_bit_cast(vec8, __builtin_amdgcn_raw_buffer_load_b128(kr_rs, off + t * 32, 0, 0));
            return;
        }
        const __amdgpu_buffer_rsrc_t rs = table(tail, kp, kc);
#pragma unroll
        for (int t = 0; t < KT; ++t) kf[t] = ld_frag(rs, row * kBlockBytes, mt * KT + t);
    };
    auto load_v = [&](bool tail, int row, int mt) {
        if constexpr (DIRECT) {
            const int off = (row * kBlock + mt * 32 + 4 * half) * v_row + col * MD * 2;
#pragma unroll
            for (int ss = 0; ss < 2; ++ss)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int at = off + (16 * ss + 8 * (e >> 2) + (e & 3)) * v_row;
                    if constexpr (MD == 2) {
                        vr[ss][e][0] = __builtin_amdgcn_raw_buffer_load_b32(vr_rs, at, 0, 0);
                    } else {
                        const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(vr_rs, at, 0, 0);
                        vr[ss][e][0] = x[0];
                        vr[ss][e][MD / 2 - 1] = x[1];
                    }
                }
            return;
        }
        const __amdgpu_buffer_rsrc_t rs = table(tail, vp, vc);
#pragma unroll
        for (int md = 0; md < MD; ++md)
#pragma unroll
            for (int ss = 0; ss < 2; ++ss) vf[md][ss] = ld_frag(rs, row * kBlockBytes, md * 4 + 2 * mt + ss);
    };
    // Centroid chunks get their score bias (log2 of the block's length over c,
    // -inf for selected blocks and padding) from one more MFMA per query tile:
    // lane (0, col) of the A operand holds centroid col's bias as bf16 parts,
    // the B operand ones in those slots.  bf16 for both input types (bias / c
    // can exceed fp16's range at small softmax scales); three parts carry the
    // fp32 value exactly.
    bf16x8 ones_frag;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones_frag[e] = (bf16_t)((half == 0 && e < 3) ? 1.0f : 0.0f);
    auto bias_frag = [&](int row, int mt) -> bf16x8 {
        bf16x8 f;
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = (bf16_t)0.0f;
        const uint32_t word = (2 * row + mt < a.mask_words) ? my_mask[2 * row + mt] : 0u;
        const int j = row * kBlock + mt * 32 + col;
        const bool dead = ((word >> col) & 1u) != 0u || j >= a.centroids;
        const float b = (j == a.centroids - 1 ? a.last_len_log2 : 6.0f) * a.inv_scale_log2;
        const bf16_t b0 = (bf16_t)b;
        const float r1 = b - (float)b0;
        const bf16_t b1 = (bf16_t)r1;
        if (half == 0) {
            f[0] = dead ? (bf16_t)(-__builtin_inff()) : b0;
            f[1] = dead ? (bf16_t)0.0f : b1;
            f[2] = dead ? (bf16_t)0.0f : (bf16_t)(r1 - (float)b1);
        }
        return f;
    };
    // scores of half mt of the chunk in table row `row` (its key fragments are in kf)
    auto scores = [&](f32x16 (&s)[NT], bool tail, int row, int mt) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int v = 0; v < 16; ++v) s[nt][v] = 0.0f;
        if constexpr (DIRECT) {
            if (!all_dims) {  // what lies past a narrower row must not meet the zero query dims
#pragma unroll
                for (int t = 0; t < KT; ++t)
                    if (t * 16 + half * 8 >= a.head_dim) kf[t] = vec8(T(0.0f));
            }
        }
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) s[nt] = mfma32(kf[t], qreg[nt][t], s[nt]);
        if (TAIL && tail) {
            const bf16x8 b = bias_frag(row, mt);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) s[nt] = mfma32(b, ones_frag, s[nt]);
        }
    };
    auto pv = [&](const vec8 (&pf)[NT][2]) {
#pragma unroll
        for (int ss = 0; ss < 2; ++ss)
#pragma unroll
            for (int md = 0; md < MD; ++md) {
                vec8 f;
                if constexpr (DIRECT) {  // element md of the 8 keys
                    u32x4 w;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        w[j] = __builtin_amdgcn_perm(vr[ss][2 * j + 1][md / 2], vr[ss][2 * j][md / 2],
                                                     md % 2 ? 0x07060302u : 0x05040100u);
                    f = __builtin_bit_cast(vec8, w);
                } else {
                    f = vf[md][ss];
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) o[md][nt] = mfma32(f, pf[nt][ss], o[md][nt]);
            }
    };
    // column maxima and running-max update of half mt of a chunk; `plain`: an
    // exact full block, else a short last key block is masked first
    auto check = [&](f32x16 (&s)[NT], bool tail, int row, int mt, bool plain) {
        if (!plain && !tail && (row + 1) * kBlock > a.kv_tokens) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                if (row * kBlock + mt * 32 + 8 * (v >> 2) + 4 * half + (v & 3) >= a.kv_tokens)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) s[nt][v] = -__builtin_inff();
        }
        float mx[NT];
        half_max<NT>(s, c, mx);
        rescale_to<NT, MD>(mx, true, nm, mth, l, lt, o);
    };

    f32x16 sa[NT], sb[NT];  // scores of the first / second half of the current chunk
    int row0 = table_row(lo), row1 = table_row(lo + 1);
    load_k(is_tail(lo), row0, 0);
    load_v(is_tail(lo), row0, 0);
    scores(sa, is_tail(lo), row0, 0);
    load_k(is_tail(lo), row0, 1);
    check(sa, is_tail(lo), row0, 0, false);
    // One chunk: its first half's softmax and PV product beside the scores of
    // its second half, then the second half's beside the scores of the next
    // chunk.  `last` (no next chunk) and `plain` (this chunk and the next are
    // exact full blocks) are constants of each inlined copy.
    auto chunk_step = [&](int cc, bool last, bool plain, bool half0_only) __attribute__((always_inline)) {
        const int row2 = (plain && !SPARSE) ? cc + 2 : table_row(cc + 2);
        const bool t0 = !plain && is_tail(cc), t1 = !plain && !last && is_tail(cc + 1);
        vec8 pf[NT][2];
        if (!half0_only) scores(sb, t0, row0, 1);
        if (!last) load_k(t1, row1, 0);
        probs_half<T, NT>(sa, c, nm, l, lt, t0, pf);
        pv(pf);
        if (!half0_only) {
            load_v(t0, row0, 1);
            check(sb, t0, row0, 1, plain);
        }

        if (!last) {
            scores(sa, t1, row1, 0);
            load_k(t1, row1, 1);
        }
        if (!half0_only) {
            probs_half<T, NT>(sb, c, nm, l, lt, t0, pf);
            pv(pf);
        }
        if (!last) {
            load_v(t1, row1, 0);
            check(sa, t1, row1, 0, plain);
        }
        row0 = row1;
        row1 = row2;
    };
    // the selection is ascending, so only the last exact chunk can be short
    int cc = lo;
    for (; cc + 3 <= n_exact && cc + 1 < hi; ++cc) chunk_step(cc, false, true, false);
    for (; cc + 1 < hi; ++cc) chunk_step(cc, false, false, false);
    // A last centroid chunk whose second half is only padding ends after its
    // first (the rest would add exactly zero to l, l_tail and O).
    chunk_step(cc, true, false, TAIL && hi == n_chunks && row0 * kBlock + 32 >= a.centroids);

    // ---- merge of the W parts, first-order correction, store
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        l[nt] = add_xor32(l[nt]);
        lt[nt] = add_xor32(lt[nt]);
    }
    // output units, kUnits / W per wave: (tile, pair of 4-row accumulator groups), or
    // DIRECT one group over all tiles (its 4 MD values are consecutive dims)
    constexpr int kUnits = DIRECT ? NT * 4 : MD * NT * 2;
    __shared__ __attribute__((aligned(16))) float parts[W > 1 ? W * MD * NT * 16 * 64 : 4];
    __shared__ float stat[W > 1 ? W : 1][3][kBlock];
    if constexpr (W > 1) {
        float m[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            m[nt] = mth[nt] == -__builtin_inff() ? -__builtin_inff() : -nm[nt];
            if (half == 0) {
                stat[wave][0][32 * nt + col] = m[nt];
                stat[wave][1][32 * nt + col] = l[nt];
                stat[wave][2][32 * nt + col] = lt[nt];
            }
        }
        __syncthreads();
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float top = -__builtin_inff();
#pragma unroll
            for (int w = 0; w < W; ++w) top = fmaxf(top, stat[w][0][32 * nt + col]);
            auto factor = [&](float mw) { return mw == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(mw - top); };
            l[nt] = 0.0f;
            lt[nt] = 0.0f;
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const float f = factor(stat[w][0][32 * nt + col]);
                l[nt] += stat[w][1][32 * nt + col] * f;
                lt[nt] += stat[w][2][32 * nt + col] * f;
            }
            const float f = factor(m[nt]);
#pragma unroll
            for (int md = 0; md < MD; ++md)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    f32x4 x;
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[e] = o[md][nt][4 * g + e] * f;
                    *reinterpret_cast<f32x4*>(&parts[((((wave * MD + md) * NT + nt) * 4 + g) * 64 + lane) * 4]) = x;
                }
        }
        __syncthreads();
    }
    const bool first_order = TAIL && a.ht != nullptr;
    const __amdgpu_buffer_rsrc_t ht_rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(first_order ? a.ht + (int64_t)bh * D * D * 2 : a.kp), (short)0, first_order ? D * D * 2 : 0,
        kRawFlags);
    typedef T vec4 __attribute__((ext_vector_type(4)));
    // 16-byte stores when every output row start is 16-byte aligned (8-byte ones otherwise)
    const bool st16 = (reinterpret_cast<uintptr_t>(a.o.data) % 16 == 0) &&
                      ((a.o.sb | a.o.sh | a.o.st) * (int64_t)sizeof(T)) % 16 == 0;
#pragma unroll
    for (int u = 0; u < kUnits / W; ++u) {
        // W = 1: tile and pair are constants and the accumulators stay in registers
        const int unit = wave * (kUnits / W) + u;
        const int p = unit & 1, nt = DIRECT ? unit >> 2 : (unit >> 1) & 1, md = DIRECT ? 0 : unit >> 2;
        const bool second = nt != 0;
        constexpr int kVals = DIRECT ? 4 * MD : 8;
        float x[kVals];
        if constexpr (DIRECT) {
            const int g = unit & 3;
#pragma unroll
            for (int d = 0; d < MD; ++d) {
                f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (W > 1) {
#pragma unroll
                    for (int w = 0; w < W; ++w)
                        sum += *reinterpret_cast<const f32x4*>(&parts[((((w * MD + d) * NT + nt) * 4 + g) * 64 + lane) * 4]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[e] = o[d][u >> 2][4 * (u & 3) + e];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) x[MD * e + d] = sum[e];
            }
        } else if constexpr (W > 1) {
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int w = 0; w < W; ++w)
                    sum += *reinterpret_cast<const f32x4*>(
                        &parts[((((w * MD + md) * NT + nt) * 4 + 2 * p + g) * 64 + lane) * 4]);
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * g + e] = sum[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = o[u >> 2][(u >> 1) & 1][8 * (u & 1) + e];
        }
        const float lf = second ? l[1] : l[0];
        const float inv = 1.0f / lf;
#pragma unroll
        for (int e = 0; e < kVals; ++e) x[e] *= inv;
        if (first_order) {
            // rows 32md .. of the packed D x D matrix (kfrag_elem) times the query tile
            f32x16 corr;
#pragma unroll
            for (int v = 0; v < 16; ++v) corr[v] = 0.0f;
#pragma unroll
            for (int t = 0; t < KT; ++t) {
                // element by element: a choice between the arrays' elements puts them in private memory
                const u32x4 q0 = __builtin_bit_cast(u32x4, qreg[0][t]), q1 = __builtin_bit_cast(u32x4, qreg[1][t]);
                u32x4 qt;
#pragma unroll
                for (int j = 0; j < 4; ++j) qt[j] = second ? q1[j] : q0[j];
                corr = mfma32(ld_frag(ht_rs, md * KT * 1024, t), __builtin_bit_cast(vec8, qt), corr);
            }
            const float wa = (second ? lt[1] : lt[0]) * inv * a.corr_scale;
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] += (p ? corr[8 + e] : corr[e]) * wa;
        }
        const int tok = qbase + (second ? q_off[1] : q_off[0]);
        if (tok >= a.q_tokens) continue;  // lanes l and l + 32 (one query) take the same branch
        char* dst = a.o.data + a.o.row(bh, tok) * (int64_t)sizeof(T);
        u32x2 w4[kVals / 4];  // w4[g]: dims 32md + 8(2p + g) + 4half ..; DIRECT: MD (8g' + 4half) + 4g .. of group g'
#pragma unroll
        for (int g = 0; g < kVals / 4; ++g) {
            vec4 out;
#pragma unroll
            for (int e = 0; e < 4; ++e) out[e] = from_f32<T>(x[4 * g + e]);
            w4[g] = __builtin_bit_cast(u32x2, out);
        }
        if constexpr (DIRECT) {
#pragma unroll
            for (int j = 0; j < MD / 2; ++j) {
                const int d = MD * (8 * (unit & 3) + 4 * half) + 8 * j;
                if (d >= a.head_dim) continue;
                char* to = dst + d * sizeof(T);
                if (st16) {
                    *reinterpret_cast<u32x4*>(to) =
                        u32x4{w4[2 * j][0], w4[2 * j][1], w4[2 * j + 1][0], w4[2 * j + 1][1]};
                } else {
                    *reinterpret_cast<u32x2*>(to) = w4[2 * j];
                    *reinterpret_cast<u32x2*>(to + 8) = w4[2 * j + 1];
                }
            }
            continue;
        }
        if (st16) {
            // one lane-half swap per dword leaves lanes 0-31 with dims 8(2p) .. +7 and
            // lanes 32-63 with dims 8(2p + 1) .. +7 of the tile
            u32x4 x16;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const auto r = __builtin_amdgcn_permlane32_swap(w4[0][j], w4[1][j], false, false);
                x16[j] = r[0];
                x16[2 + j] = r[1];
            }
            const int d = md * 32 + 8 * (2 * p + half);
            if (d < a.head_dim) *reinterpret_cast<u32x4*>(dst + d * sizeof(T)) = x16;
        } else {
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                const int d = md * 32 + 8 * (2 * p + g) + 4 * half;
                if (d < a.head_dim) *reinterpret_cast<u32x2*>(dst + d * sizeof(T)) = w4[g];
            }
        }
    }
}

// SIMDs of the device (0 if it does not say).
int simd_count() {
    static const int simds = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        return 4 * cus;
    }();
    return simds;
}

// Waves per query block: the W with the smallest estimate of
//     rounds of the SIMDs x (chunks of one wave + the chunk times a merge costs),
// which follows the measured times (1280 blocks of 64 chunks, [2,10,4096,64]:
// 126 / 108 / 98 / 122 us at W = 1 / 2 / 4 / 8, estimates 130 / 107 / 98 / 125;
// 2048 such blocks: 142 / 145 / 148 / 184 us, estimates 130 / 142 / 156 / 200;
// 128 blocks of 16 chunks: 17.7 us with one wave, under 12 with 2, 4 or 8).  A
// grid that leaves SIMDs idle, or its last round nearly empty, is split; a full
// one keeps one wave per block and merges nothing.  Eight waves use 134 KB of
// LDS, one workgroup per CU, so nothing runs beside their merge.
int waves_per_block(int64_t blocks, int n_chunks, int most) {
    const int simds = simd_count();
    if (simds <= 0) return 1;
    int best = 1;
    double least = 0.0;
    for (int w = 1; w <= most && w <= n_chunks; w *= 2) {
        const double merge = w == 1 ? 1.0 : w == 8 ? 4.5 : 3.5;
        const double cost = (double)((blocks * w + simds - 1) / simds) * ((n_chunks + w - 1) / w + merge);
        if (w == 1 || cost < least) {
            best = w;
            least = cost;
        }
    }
    return best;
}

template <typename T, int D, bool SPARSE, bool TAIL, bool DIRECT>
int launch_t(const AttnArgs& a, const KvRows& kv, int bh_count, hipStream_t stream) {
    const int blocks = bh_count * a.q_blocks;
    const int n_chunks = (SPARSE ? a.exact : a.kv_blocks) + (TAIL ? a.npad / kBlock : 0);
    constexpr int kMost = D <= 64 ? 8 : 4;  // waves of a workgroup: two per SIMD, one at D = 128
    const int w = waves_per_block(blocks, n_chunks, kMost);
#define PISA_PARTS(W)                                                                                              \
    hipLaunchKernelGGL((attention_parts_kernel<T, D, SPARSE, TAIL, W, DIRECT>), dim3(blocks), dim3(64 * W), 0, stream, \
                       a, kv, a.idx, a.selmask)
    if (w == 1) PISA_PARTS(1);
    else if (w == 2) PISA_PARTS(2);
    else if (w == 4) PISA_PARTS(4);
    else if constexpr (kMost == 8) PISA_PARTS(8);
#undef PISA_PARTS
    return pisa_host::check_launch("attention_parts_kernel");
}

}  // namespace

// At most one wave per SIMD, from packed tables: nothing then hides the loads of
// the kernel above, and the one of attention.hip, whose 264 registers hold both
// halves' fragments, is the faster one.  Call times, this kernel -> that one:
// [1,14,2880,64] 57.4 -> 54.5 us, 2048 keys of 4096 tokens in 12 heads 41.1 ->
// 39.3, [1,11,4630,64] 86.8 -> 82.6, [1,8,8192,64] 150.3 -> 146.7, [1,32,2048,64]
// 52.0 -> 51.2.  Splits and grids of more than a round stay here ([1,16,2048,64],
// two waves per block, 39.0 against 39.5; 2808 blocks of 11 chunks 48.7 against
// 50.2).
bool dense_d64_one_wave(const AttnArgs& a, int bh_count) {
    const int64_t blocks = (int64_t)bh_count * a.q_blocks;
    return blocks <= simd_count() && waves_per_block(blocks, a.kv_blocks, 8) == 1;
}

int launch_attention_d64(int dtype, bool sparse, const AttnArgs& a, int bh_count, hipStream_t stream) {
    const KvRows none{};
    if (dtype == PISA_DTYPE_BF16)
        return sparse ? launch_t<bf16_t, 64, true, true, false>(a, none, bh_count, stream)
                      : launch_t<bf16_t, 64, false, false, false>(a, none, bh_count, stream);
    return sparse ? launch_t<f16_t, 64, true, true, false>(a, none, bh_count, stream)
                  : launch_t<f16_t, 64, false, false, false>(a, none, bh_count, stream);
}

// Reading rows in place saves the packing launch (about 4.5 us and 6.7 ns a key
// block at width 64) and costs 0.05 to 0.1 us, more at 128, for every chunk that
// the busiest CU walks: `load` below, which a grid of a few blocks, or of a few
// blocks over a whole round, makes larger than its share of all chunks.  So the
// lines are in `load` and key blocks (`tables`), one for each kernel that the
// packed call would run and each way the rows lie in memory, under bounds in all
// chunks.  They were fitted to the device times of 130 calls of 2 to 48 heads in
// three layouts ([B,H,T,D], [B,T,H,D] and a fused projection) at head dims 40, 64,
// 80, 96, 104 and 128 on one MI355X.  Packed / in place, us:
//   width 64, at most one wave per SIMD (dense_d64_one_wave, the better packed
//     kernel of the two): [1,24,2048,64] 43.1 / 42.7, 2048 keys of 4096 tokens in
//     12 heads 39.4 / 42.7; as [B,T,H,D] rows [1,24,1536,64] 33.5 / 36.4 and at
//     head dim 40 [1,24,2048] 41.9 / 47.1.  Otherwise [1,16,2048,64] 39.0 / 36.6,
//     16384 keys of 256 tokens in 2 heads 67.6 / 78.6, [2,24,9216,64] x 77
//     34.9 / 33.6.
//   width 128 splits small grids where the packed kernel does not.  Up to a
//     quarter of a round in place always wins ([1,8,2048,128] 35.1 / 28.5); up to
//     half a round it wins against the kernel of uneven grids ([2,15,940,128]
//     39.3 / 28.5), and against the persistent one the more of the SIMDs its two
//     waves per block fill ([1,16,2048,128] 51.9 / 49.8, [2,8,1374,128] 33.1 /
//     35.9, [1,8,3072,128] 57.2 / 69.9); above, its chunks cost half as much again
//     ([1,16,9216,128] x 256 38.9 / 46.8, [2,20,1024,128] 42.2 / 38.7).
//   padded width 96 runs on the kernel of 128 in place, and on one that neither
//     splits nor persists packed: [1,8,4096,80] 84.9 / 70.7, [1,24,1536,80]
//     42.6 / 45.9.  Rows that are not whole 128-byte lines but lie a multiple of
//     them apart ([B,T,H,D] with 8 heads of 80) cost a quarter more each:
//     [1,8,3072,80] 65.4 / 69.2, against 75.0 / 65.1 for [1,7,3373,80].
// The rows of a head, rounded up to whole chunks, are addressed with 32-bit byte
// offsets.
bool dense_rows_in_place(int padded, const AttnArgs& a, const KvRows& kv, int bh_count) {
    if (padded > 128) return false;
    auto addressable = [&](const View& x) { return x.st > 0 && x.st <= INT32_MAX / 2 / ((int64_t)a.kv_blocks * kBlock + 1); };
    if (!addressable(kv.k) || !addressable(kv.v)) return false;
    const int64_t blocks = (int64_t)bh_count * a.q_blocks, tables = (int64_t)bh_count * a.kv_blocks;
    const int64_t chunks = blocks * a.kv_blocks;
    const int64_t simds = simd_count() > 0 ? simd_count() : 1024;
    const int64_t load = (blocks + simds / 4 - 1) / (simds / 4) * a.kv_blocks;
    const bool joined = kv.k.st == a.head_dim && kv.v.st == a.head_dim;  // one row right after the other
    if (padded == 64) {
        if (chunks >= 13000 + 19 * tables) return false;
        if (dense_d64_one_wave(a, bh_count))
            return 100 * load < (a.head_dim < 64 ? 1300 + 5 * tables : joined ? 4600 + 7 * tables : 1400 + 7 * tables);
        return waves_per_block(blocks, a.kv_blocks, 8) == 1 || 200 * load < 6000 + 27 * tables;
    }
    if (padded == 128 ? chunks >= 9500 + 14 * tables : blocks > simds / 2 && chunks >= 7000 + 20 * tables) return false;
    if (blocks <= simds / 4) return true;
    const bool persistent = a.head_dim == 128 && blocks % 8 == 0;  // the packed kernel (launch_attention_t)
    if (blocks <= simds / 2) {
        const bool lines_apart = a.head_dim % 64 != 0 && (kv.k.st % 64 == 0 || kv.v.st % 64 == 0);
        return !(persistent || lines_apart) || 100 * load < 600 + 23 * tables * blocks / simds;
    }
    if (padded == 96) return 100 * load < 800 + (joined ? 8 : 4) * tables;
    return 200 * load < 2400 + (joined && a.head_dim < 128 ? 40 : persistent ? 13 : 16) * tables;
}

int launch_attention_rows(int dtype, int padded, const AttnArgs& a, const KvRows& kv, int bh_count, hipStream_t stream) {
    if (padded == 64)
        return dtype == PISA_DTYPE_BF16 ? launch_t<bf16_t, 64, false, false, true>(a, kv, bh_count, stream)
                                        : launch_t<f16_t, 64, false, false, true>(a, kv, bh_count, stream);
    return dtype == PISA_DTYPE_BF16 ? launch_t<bf16_t, 128, false, false, true>(a, kv, bh_count, stream)
                                    : launch_t<f16_t, 128, false, false, true>(a, kv, bh_count, stream);
}

}  // namespace pisa
