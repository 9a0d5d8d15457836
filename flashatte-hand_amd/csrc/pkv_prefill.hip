// pkv_prefill.hip — attention of many query rows per KV head over the paged
// cache (prefill chunks, long verify steps) on gfx950.
//
// The decode partition kernels give a wave its own K/V tile, which suits one
// to a few dozen query rows per KV head: the cache is read once and the call
// is bound by HBM.  With hundreds of rows the call is bound by the matrix
// cores and by the softmax between the two products, and every wave staging
// its own copy of the same tile makes the LDS and the L2 the limit instead.
// Here a workgroup of 4 waves takes kRows = 128 query rows of one
// (b, KV head) and stages each K/V tile once for all of them.
//
//   rows    wave w holds rows 32 w .. 32 w + 31 of the block: Q^T in VGPRs as the
//           B operand of v_mfma_f32_32x32x16_{bf16,f16} (lane (n, h): row n,
//           dims 16 kk + 8 h .. + 7), O^T and the softmax state in VGPRs.
//   tile    64 tokens of K and V, two LDS buffers: the next tile's rows go straight
//           into the other buffer (global_load_lds, 16 bytes per lane; FP8 rows
//           through registers, converted) while this one is used, one barrier per
//           tile.  Page ids are loaded a tile further ahead, so no K/V address
//           waits for the block table.
//   QK      S^T[32 tok x 32 rows] = K Q^T.  Lane (n, h) of the result holds row
//           n, tokens 8 a + 4 h + c (a, c < 4): every lane has one query row, so
//           the row maximum and sum need one cross-lane step.
//   PV      O^T[D x 32 rows] += V^T P^T over 16 tokens a step, in the token
//           order the scores already have: the k index 8 h + e of the operands
//           stands for token 8 (e / 4) + 4 h + e % 4 of the step, so P^T is used
//           in place and V^T comes from ds_read_b64_tr_b16 with the same order.
//           The fp32 probabilities go in as a 16-bit head and a 16-bit
//           remainder (two products per V^T operand), as in the decode kernels.
//   order   a pipeline over blocks of 32 tokens, in slots of one matrix product
//           each (24 at head_dim 128): the scores of the next block, the softmax
//           of this one and the PV product of the last one are independent, so
//           a wave issues its softmax, operand reads and loads while its own
//           products run.  The slots are fixed with scheduling barriers: left to
//           the compiler, the probabilities sank behind the products.
//
// Bound: the matrix cores and their power.  Over 16,384 tokens of context (4 x 512
// query tokens, 32/8 heads, head_dim 128) 727-735 TFLOP/s counted without the
// remainders' products, 1,090-1,100 with them, while the clock falls to about
// 1.7 GHz; a large bf16 matrix product reaches 1,190 on the same card.  The
// decode kernels took 1,892 us for that call, this one 767; 4 x 512 over 0-4,096 tokens
// 304 against 135 (135-142 on several cards, append and merge included).  Steps on the way, each
// in its own run (4 x 512 over 0-4,096): waiting for the page
// ids where they were loaded 171 us, not 157; padded rows and loads through
// registers 155; the next tile's loads in a burst and not spread over the slots
// +15 (a load waits for the one before it at 64 bytes a clock and CU); rows
// stored from registers and not through the LDS +11.
//
// Work is dealt as in the decode's tile schedule, in units of 64-token tiles:
// a stream is the tiles that one (b, KV head, row block) can see (a causal
// block of early queries is shorter than a late one), streams are laid end
// to end and every workgroup takes an equal share of units.  A stream inside
// one share goes straight to the output; a share's cut streams leave fp32
// partials that prefill_combine_kernel merges.
#include <utility>

#include "pkv_partition_impl.h"

namespace pkv {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kRows = kPrefillRows;
constexpr int kThreads = 256;
constexpr int kPrefillTok = 64;   // tokens per tile
constexpr int kPrefillSnap = 2;   // units within which a share's end moves to a stream's edge

template <bool BF16>
__device__ __forceinline__ f32x16 mfma_32x32x16(const uint4& a, const uint4& b, f32x16 c) {
    if constexpr (BF16) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                      0, 0, 0);
    }
}

// f(0), f(1), ... f(N - 1), each index a compile-time constant.
template <int... I, typename F>
__device__ __forceinline__ void unrolled_over(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
    unrolled_over(std::make_integer_sequence<int, N>{}, f);
}

// The 16-bit remainders of two fp32 values whose rounded heads are packed in
// `heads`: value - head is exact in fp32 (Sterbenz), taken in one instruction
// with the head picked out of the pair (bf16: a two-element dot product with
// (-1, 0) or (0, -1); fp16: a mixed-precision FMA).
template <bool BF16>
__device__ __forceinline__ uint32_t remainder2(uint32_t heads, float p0, float p1, uint32_t minus_lo,
                                               uint32_t minus_hi) {
    if constexpr (BF16) {
        return pack2_hw<true>(dot2<true>(heads, minus_lo, p0), dot2<true>(heads, minus_hi, p1));
    } else {
        return pack2_hw<false>(fmaf(f16_lo(heads), -1.f, p0), fmaf(f16_hi(heads), -1.f, p1));
    }
}

// The first key that some row of block `hg` can see in a row of `seqlen` tokens.
// Window bounds are taken in 64 bits (a window near INT32_MAX must not wrap).
__device__ __forceinline__ int32_t first_visible(const PartitionParams& p, int32_t seqlen, int32_t hg) {
    if (p.win_left < 0) {
        return 0;
    }
    const int64_t lo = static_cast<int64_t>(seqlen) - p.q_len + hg * kRows / p.group - p.win_left;
    return static_cast<int32_t>(min(max(lo, int64_t{0}), static_cast<int64_t>(seqlen)));
}

// Tiles of a stream: the 64-token tiles some row of block `hg` can see in a
// row of `seqlen` tokens.
__device__ __forceinline__ TileSpan prefill_span(const PartitionParams& p, int32_t seqlen, int32_t hg) {
    const int32_t r1 = min(p.rows, (hg + 1) * kRows) - 1;
    const int32_t lo = first_visible(p, seqlen, hg);
    int64_t hi = seqlen;
    if (p.win_right >= 0) {
        hi = static_cast<int64_t>(seqlen) - p.q_len + r1 / p.group + p.win_right + 1;
        hi = min(max(hi, int64_t{0}), static_cast<int64_t>(seqlen));
    }
    TileSpan t;
    t.first = lo / kPrefillTok;
    t.n = hi > lo ? static_cast<int32_t>((hi + kPrefillTok - 1) / kPrefillTok) - t.first : 0;
    return t;
}

// A cut stream, written by the workgroup that owns its first tile: the
// combine merges partial slots 2 w + 1, 2 (w + 1), 2 (w + 2), ... (`parts` of
// them).  parts == 0: nothing to merge.
struct CutStream {
    int32_t parts;
    int32_t b;
    int32_t kvh;
    int32_t hg;
};

template <bool BF16, int D, bool FP8>
struct Prefill {
    static constexpr int kTok = kPrefillTok;
    static constexpr int KK = D / 16;      // MFMA steps of one QK product
    static constexpr int DT = D / 32;      // O^T tiles of 32 dims
    static constexpr int CH = D / 8;       // 16-byte chunks per token row
    static constexpr int RP = kThreads / CH; // token rows per load pass
    static constexpr int NP = kTok / RP;   // passes per tile and tensor
    static constexpr int RW = 64 / CH;     // token rows of a pass per wave
    static constexpr int EB = FP8 ? 1 : 2;
    static constexpr int kBuf = kTok * D;  // elements of one LDS tile
    static constexpr float kProbLog2Offset = BF16 ? 0.f : 7.f; // as in MfmaMath
    using Chunk = typename TileRegs<64, FP8>::Chunk;
    // Dims of O^T tile dt: index m < 16 is dim dim0(dt) + m, m >= 16 is dim
    // dim0(dt) + kSplit + m - 16.
    static constexpr int kSplit = D == 64 ? 32 : 64;
    static __device__ constexpr int dim0(int dt) { return D == 256 ? 16 * (dt & 3) + 128 * (dt >> 2) : 16 * dt; }
    // Rows are unpadded (the direct loads write 64 lanes x 16 bytes in a row), so
    // chunk c of row r sits at place c ^ swz(r): the 16 rows that a K operand
    // read touches at one chunk, and the 4 rows x 2 x 32 bytes of half a V^T
    // read, fall on all 64 banks once.
    static constexpr uint32_t kFlip8 = D == 64 ? 64 : 16; // 16 (swz(r + 8) ^ swz(r)), r & 8 == 0
    static __device__ int swz(int r) {
        if constexpr (D == 64) {
            return (r & 2) | ((r >> 2) & 1) | ((r >> 1) & 4);
        } else {
            return ((r & 7) << 1) | ((r >> 3) & 1);
        }
    }
};

// 16 bytes per lane from base + off straight into LDS at lds + 16 * lane
// (wave-uniform base and lds).  Counted by vmcnt, which the compiler does not
// know here: dma_wait() before the barrier that publishes the tile.  It writes
// a buffer that nobody reads before that barrier, so reads may pass it.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm" // m0 is a reserved register: its clobber is declared all the same
__device__ __forceinline__ void dma16(uint64_t base, uint32_t off, uint32_t lds) {
    // Five wait states: base may come from a lane read just before.
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(off), "s"(base)
                 : "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }

typedef __attribute__((address_space(3))) uint16_t lds_u16;

template <bool BF16, int D, bool FP8, bool CAP>
__global__ __launch_bounds__(kThreads, D == 256 ? 1 : 2) void prefill_kernel(PartitionParams p) {
    using C = Prefill<BF16, D, FP8>;
    constexpr int kTok = C::kTok;
    // Tiles K 0, K 1, V 0, V 1.
    __shared__ __attribute__((aligned(1024))) uint16_t smem[4 * C::kBuf];

    const int tid = threadIdx.x;
    const int wave = uniform(tid >> 6);
    const int lane = tid & 63;
    const int n = lane & 31;
    const int h = lane >> 5;
    const int nhg = p.head_groups;
    const int hk = p.num_heads_k;

    // Workgroup i runs on XCD i mod 8: neighbouring shares (the row blocks of
    // one KV head, which read the same K/V) go to one XCD and its L2.
    const int launched = p.tile_workers;
    const int xcd = static_cast<int>(blockIdx.x) & 7;
    const int w = xcd * (launched >> 3) + min(xcd, launched & 7) + (static_cast<int>(blockIdx.x) >> 3);
    CutStream* const cuts = reinterpret_cast<CutStream*>(p.part_lse + static_cast<int64_t>(launched) * 2 * kRows);

    // ---- plan: the prefix of the row blocks' units (one KV head), in the
    // order (row, block); every KV head of a row repeats the row's units.
    const auto row_len = [&](int b) { return min(max(p.seqlens[b], 0), p.row_cap); };
    const int entries = p.batch * nhg; // <= kPrefillEntries (host rule)
    uint32_t* const prefix = reinterpret_cast<uint32_t*>(smem);
    uint32_t* const scratch = prefix + kPrefillEntries + 1;
    {
        const int per = (entries + kThreads - 1) / kThreads;
        const int e0 = tid * per;
        const int e1 = min(e0 + per, entries);
        int eb = e0 / nhg;
        int eg = e0 - eb * nhg;
        int sl = row_len(min(eb, p.batch - 1));
        uint32_t mine = 0;
        for (int e = e0; e < e1; ++e) {
            prefix[e] = mine;
            mine += prefill_span(p, sl, eg).n + kPrefillHeader;
            if (++eg == nhg && e + 1 < e1) {
                eg = 0;
                sl = row_len(++eb);
            }
        }
        const uint32_t incl = wave_inclusive_scan_u32(mine);
        if (lane == 63) {
            scratch[wave] = incl;
        }
        __syncthreads();
        uint32_t before = incl - mine;
        for (int k = 0; k < wave; ++k) {
            before += scratch[k];
        }
        for (int e = e0; e < e1; ++e) {
            prefix[e] += before;
        }
        if (tid == 0) {
            prefix[entries] = scratch[0] + scratch[1] + scratch[2] + scratch[3];
        }
        __syncthreads();
    }
    const uint32_t total = uniform(static_cast<int32_t>(prefix[entries])) * static_cast<uint32_t>(hk); // < 2^31 (host rule)
    // Workgroups with a share.  The launch is sized from max_seqlen, and rows may
    // be far shorter; a smaller share then cuts the streams into more parts than
    // their merge is worth.  With u units per stream a share has at least
    // sqrt(u) / 4 units, and 3 where that still leaves one workgroup per CU.  Measured
    // (head_dim 64, 8 query tokens x 16 heads per KV head, table of 131,072 tokens; shares
    // of one unit or more / this / the decode kernels, us): 8 streams of 64 tiles 32 / 28 /
    // 22.5, 2 of 256 tiles 46 / 28 / 21, 32 of 16 tiles 30 / 26 / 22.7.
    const float per_stream = static_cast<float>(total) / static_cast<float>(entries * hk);
    const float most = fminf(static_cast<float>(launched),
                             fmaxf(static_cast<float>(kComputeUnits), static_cast<float>(total) * (1.f / 3.f)));
    const float least = fmaxf(1.f, 0.25f * sqrtf(per_stream)); // units per share
    const int32_t workers = uniform(max(1, static_cast<int32_t>(fminf(most, static_cast<float>(total) / least))));
    if (w >= workers) {
        if (tid == 0) {
            cuts[w] = CutStream{0, 0, 0, 0};
        }
        return;
    }
    // Share w: units [w T / W, (w + 1) T / W), each quotient in 32 bits.
    const auto share = [&](int i) {
        const uint32_t quot = total / static_cast<uint32_t>(workers);
        const uint32_t rem = total - quot * static_cast<uint32_t>(workers);
        return static_cast<int32_t>(static_cast<uint32_t>(i) * quot +
                                    static_cast<uint32_t>(i) * rem / static_cast<uint32_t>(workers));
    };
    // Both ends of the share, moved to a stream's edge where they fall within
    // kPrefillSnap units of it.  For each, the thread whose entry holds the unit
    // says which stream it is in.
    int x0 = share(w);
    int x_end = share(w + 1);
    for (int e = tid; e < entries; e += kThreads) {
        const int eb = e / nhg;
        const int row0 = static_cast<int>(prefix[eb * nhg]);
        const int units = static_cast<int>(prefix[(eb + 1) * nhg]) - row0;
        const int at = static_cast<int>(prefix[e]) - row0;
        const int size = static_cast<int>(prefix[e + 1]) - row0 - at;
#pragma unroll
        for (int side = 0; side < 2; ++side) {
            const int rel = (side == 0 ? x0 : x_end - 1) - row0 * hk;
            if (rel >= 0 && rel < units * hk) {
                const int head = rel / units;
                const int y = rel - head * units - at;
                if (0 <= y && y < size) {
                    int* const said = reinterpret_cast<int*>(scratch) + 8 + 8 * side;
                    said[0] = eb;
                    said[1] = head;
                    said[2] = e - eb * nhg;
                    said[3] = row0 * hk + head * units + at;
                    said[4] = size;
                }
            }
        }
    }
    __syncthreads();
    const int* const said = reinterpret_cast<const int*>(scratch) + 8;
    int b = uniform(said[0]);
    int kvh = uniform(said[1]);
    int hg = uniform(said[2]);
    int vs = uniform(said[3]); // first unit of the current stream
    const auto snap = [&](int x, int from, int size) { // from <= x <= from + size
        const int to = from + size;
        if (x == to) {
            return to;
        }
        return x - from <= kPrefillSnap ? from : to - x <= kPrefillSnap ? to : x;
    };
    x0 = snap(x0, vs, uniform(said[4]));
    x_end = w + 1 == workers ? x_end : snap(x_end, uniform(said[11]), uniform(said[12]));
    const bool next_stream = x0 == vs + uniform(said[4]); // the share starts with the stream after it
    const int skip_units = uniform(said[4]);
    int seqlen = uniform(row_len(b));
    __syncthreads(); // the tiles take the LDS over
    const auto advance = [&]() {
        if (++hg == nhg) {
            hg = 0;
            if (++kvh == hk) {
                kvh = 0;
                ++b;
                seqlen = b < p.batch ? uniform(row_len(b)) : 0;
            }
        }
    };
    if (next_stream) {
        vs += skip_units;
        advance();
    }
    if (x0 >= x_end) {
        if (tid == 0) {
            cuts[w] = CutStream{0, 0, 0, 0};
        }
        return;
    }

    // remainder2's operands (-1, 0) and (0, -1), from registers: as a literal the
    // compiler writes the first as the inline constant -1.0, which the
    // instruction reads as the second.
    uint32_t minus_lo = 0x0000bf80u;
    uint32_t minus_hi = 0xbf800000u;
    asm volatile("" : "+s"(minus_lo), "+s"(minus_hi));

    // ---- the share's segments
    const uint32_t smem_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u16*)smem));
    const uint32_t smem_wave = uniform(static_cast<int32_t>(smem_at + 2u * C::RW * D * wave)); // its rows of a load pass
    const int rr = tid / C::CH;
    const int cc = tid % C::CH;
    const int pmask = (1 << p.page_shift) - 1;
    CutStream cut{0, 0, 0, 0};
    while (true) {
        const TileSpan span = prefill_span(p, seqlen, hg);
        const int units = span.n + kPrefillHeader;
        const int t_lo = max(0, x0 - vs - kPrefillHeader);
        const int t_hi = min(span.n, x_end - vs - kPrefillHeader);
        const bool empty = span.n == 0 && x0 <= vs; // no row sees a key: zeros
        if (t_lo < t_hi || empty) {
            const int tiles = t_hi - t_lo;
            int t0 = (span.first + t_lo) * kTok;
            // K/V rows of a tile.  A wave's RW rows of a load pass lie in one
            // page (P >= RW, host rule), so a pass has one wave-uniform address;
            // lane i makes that of K pass i (i < NP) or V pass i - NP, and the
            // loads read them off.
            const int32_t* __restrict__ bt_row = p.block_table + static_cast<int64_t>(b) * p.bt_stride;
            const uint32_t page_bytes = static_cast<uint32_t>(p.page_stride) * C::EB; // < 4 GiB (host rule)
            const uint32_t tok_bytes = static_cast<uint32_t>(p.token_stride) * C::EB;
            const bool v_lane = (lane & C::NP) != 0;
            const uint64_t pass_base = reinterpret_cast<uint64_t>(v_lane ? p.v : p.k) +
                                       static_cast<uint64_t>(kvh) * D * C::EB;
            const int pass_tok = C::RP * (lane & (C::NP - 1)) + C::RW * wave - (v_lane ? 32 : -32);
            // Rows past the row's end come from its last page: no query sees
            // their keys, and their V rows are cleared below.
            const int last_tok = (seqlen - 1) & ~(C::RW - 1);
            const uint32_t row_off = static_cast<uint32_t>(lane / C::CH) * tok_bytes;
            // Place cc of an LDS row holds chunk cc ^ swz(row), which depends on the
            // pass only where RP is no multiple of 16.
            const auto lane_off = [&](int pass) {
                return row_off + static_cast<uint32_t>(
                                     8 * C::EB * (cc ^ C::swz(C::RP % 16 == 0 ? rr : rr + C::RP * (pass & 1))));
            };
            int32_t ids = 0;    // page ids of the next tile's passes, as the table holds them
            uint32_t addr_lo = 0; // the passes' addresses
            uint32_t addr_hi = 0;
            // `tv`: the tile's K rows start at tv + 32, its V rows at tv - 32.
            const auto load_ids = [&](int tv) {
                ids = bt_row[min(max(tv + pass_tok, 0), last_tok) >> p.page_shift];
            };
            const auto make_addr = [&](int tv) {
                const int t = min(max(tv + pass_tok, 0), last_tok);
                const uint32_t id = static_cast<uint32_t>(ids) < static_cast<uint32_t>(p.num_pages) ? ids : 0;
                const uint64_t addr = pass_base + static_cast<uint64_t>(id) * page_bytes +
                                      static_cast<uint32_t>(t & pmask) * tok_bytes;
                addr_lo = static_cast<uint32_t>(addr);
                addr_hi = static_cast<uint32_t>(addr >> 32);
            };
            typename C::Chunk st[2 * C::NP]; // FP8 rows on their way to the LDS
            // Pass i < NP: K pass i of the tile whose K is at element `at`; else V pass i - NP.
            const auto load_pass = [&](int i, int at) {
                const int pass = i % C::NP;
                const uint64_t base = (static_cast<uint64_t>(__builtin_amdgcn_readlane(addr_hi, i)) << 32) |
                                      static_cast<uint32_t>(__builtin_amdgcn_readlane(addr_lo, i));
                if constexpr (FP8) {
                    st[i] = load_chunk<true, false>(reinterpret_cast<const char*>(base) + lane_off(pass));
                } else {
                    dma16(base, lane_off(pass),
                          smem_wave + 2u * static_cast<uint32_t>(at + (i < C::NP ? 0 : 2 * C::kBuf) + C::RP * pass * D));
                }
            };
            // The first page ids are on their way before q and the masks.
            int32_t first_ids = 0;
            if (tiles > 0) {
                load_ids(t0 - 32);
                first_ids = ids;
                load_ids(t0);
            }
            const int r_first = hg * kRows + 32 * wave;
            const int rows_here = min(32, p.rows - r_first); // <= 0: this wave has no rows
            const int r = min(r_first + n, p.rows - 1);
            const int qi = r / p.group;
            const int head = kvh * p.group + (r - qi * p.group);
            const int64_t out_row = (static_cast<int64_t>(b) * p.q_len + qi) * p.num_heads + head;
            const bool live = n < rows_here;
            const KvScales ks = kv_scales<FP8>(p, kvh);
            // The row maximum is taken before the scale, which is therefore kept
            // positive: its sign goes into q (exact).
            const float scale = fabsf(ks.score_log2);
            const uint32_t flip = ks.score_log2 < 0.f ? 0x80008000u : 0u;
            uint4 q[C::KK];
#pragma unroll
            for (int kk = 0; kk < C::KK; ++kk) {
                const uint4 v = *reinterpret_cast<const uint4*>(p.q + out_row * D + 16 * kk + 8 * h);
                q[kk] = make_uint4(v.x ^ flip, v.y ^ flip, v.z ^ flip, v.w ^ flip);
            }
            // Visible keys [lo, hi) of the lane's row, the block's first, the wave's
            // bounds, ALiBi.
            const int pad = p.kv_start != nullptr ? min(max(p.kv_start[b], 0), seqlen) : 0;
            const int first_key = uniform(max(pad, first_visible(p, seqlen, hg)));
            const int pos = seqlen - p.q_len + qi;
            int lo = first_key;
            int hi = seqlen;
            if (p.win_left >= 0) {
                lo = max(lo, static_cast<int>(max(static_cast<int64_t>(pos) - p.win_left, int64_t{0})));
            }
            if (p.win_right >= 0) {
                hi = static_cast<int>(min(static_cast<int64_t>(pos) + p.win_right + 1, static_cast<int64_t>(seqlen)));
            }
            int all_lo = live ? lo : 0;
            int all_hi = live ? hi : INT32_MAX;
#pragma unroll
            for (int d = 1; d < 32; d <<= 1) {
                all_lo = max(all_lo, __shfl_xor(all_lo, d, 64));
                all_hi = min(all_hi, __shfl_xor(all_hi, d, 64));
            }
            all_lo = uniform(all_lo);
            all_hi = uniform(all_hi);
            if (!live) {
                lo = 0;
                hi = 0;
            }
            const bool alibi = p.alibi != nullptr;
            const float slope =
                alibi ? p.alibi[static_cast<int64_t>(b) * p.alibi_stride + head] * 1.4426950408889634f : 0.f;
            const float cap = p.softcap_log2;
            const float inv_cap = CAP ? 1.f / cap : 0.f;
            const float cap_rate = -2.8853900817779268f * scale * inv_cap; // -2 log2(e) scale / cap

            f32x16 o[C::DT];
#pragma unroll
            for (int dt = 0; dt < C::DT; ++dt) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    o[dt][i] = 0.f;
                }
            }
            float m = kNegInf;
            float l = 0.f;

            // Ends the loads of K passes [kf, kt) and V passes [vf, NP): FP8 rows are converted and stored, and V rows
            // that no query of the block sees (past the row's end, padding of
            // cache_leftpad, or behind the window: the first tile may hold whole
            // pages that the caller has let go) cleared: their probability is 0,
            // but they may hold anything, and 0 times a NaN is a NaN.
            const auto finish_rows = [&](int tv, int at, int kf, int kt, int vf) {
                if constexpr (FP8) {
#pragma unroll
                    for (int i = 0; i < 2 * C::NP; ++i) {
                        const int pass = i % C::NP;
                        if (i < C::NP ? pass >= kf && pass < kt : pass >= vf) {
                            *reinterpret_cast<uint4*>(smem + at + (i < C::NP ? 0 : 2 * C::kBuf) +
                                                      (rr + C::RP * pass) * D + 8 * cc) = fp8x8_to_16<BF16>(st[i]);
                        }
                    }
                }
                if (tv - 32 < first_key || tv + 32 > seqlen) {
                    dma_wait();
#pragma unroll
                    for (int pass = 0; pass < C::NP; ++pass) {
                        const int t = tv - 32 + rr + C::RP * pass;
                        if (pass >= vf && (t < first_key || t >= seqlen)) {
                            *reinterpret_cast<uint4*>(smem + at + 2 * C::kBuf + (rr + C::RP * pass) * D + 8 * cc) =
                                make_uint4(0u, 0u, 0u, 0u);
                        }
                    }
                }
            };

            // Operands of a 32-token block (`at`: its first element in the LDS).
            // The places of a lane's chunks differ by an exclusive or of constants.
            uint32_t kaddr = smem_at + 2 * (n * D + 8 * (h ^ C::swz(n)));
            typedef short s16x4_t __attribute__((ext_vector_type(4)));
            typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
            typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
            const int vrow = 4 * h + ((lane & 15) >> 2);
            const int vdim = ((lane & 16) ? C::kSplit : 0) + 4 * (lane & 3);
            uint32_t vaddr = smem_at + 2 * (vrow * D + 8 * ((vdim >> 3) ^ C::swz(vrow)) + (vdim & 7));
            const auto read_k = [&](int at, int kk) {
                const u32x4 v = *(const lds_u32x4*)(uintptr_t)((kaddr ^ (32 * (kk & 7))) + 256 * (kk >> 3) + 2 * at);
                return make_uint4(v.x, v.y, v.z, v.w);
            };
            // V^T of dims tile dt, tokens 16 u .. 16 u + 15 of the block: half e.
            const auto read_v4 = [&](int at, int u, int dt, int e) {
                // Half 1 is eight rows on; dims from 128 on are 256 bytes on (swz moves within those).
                const uint32_t a = (vaddr ^ ((2 * C::dim0(dt) & 255) + (e ? C::kFlip8 : 0))) + (2 * C::dim0(dt) & ~255);
                return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(
                                                     a + 2 * (at + (16 * u + 8 * e) * D))));
            };
            f32x16 s[2];      // scores of an even / odd block
            uint4 ph[2][2];   // probabilities of an even / odd block: heads of its two 16-token steps
            uint4 pl[2][2];   // and their remainders
            float alpha = 1.f;
            bool raise = false;

            // The slots of one block (below).  `mul` takes the scores to log2 units.
            // With a softcap raw scores are capped first (`done`: they are already):
            // cap tanh(x / cap), tanh |y| = (1 - e) / (1 + e), e = exp(-2 |y|), times cap
            // as `mul`.  (Capped outside the slots, 4 x 512 query tokens over 2,048 with a
            // softcap took 137.7 / 175.3 us at head_dim 64 / 128, now 126.1 / 168.7;
            // without one 94 / 138.)
            const auto slots = [&](auto jc, auto bufc, bool done, float mul) {
                constexpr int j = decltype(jc)::value;
                constexpr int kat = decltype(bufc)::value * C::kBuf + j * 32 * D;
                constexpr int vat = kat + 2 * C::kBuf;
                f32x16& cur = s[j];
                f32x16& next = s[j ^ 1];
                // One basic block, in slots of one product each: what a slot
                // holds beside it (an operand read kLead slots ahead, a load pass,
                // a step of the softmax) issues while the products run.
                asm volatile("" : "+v"(kaddr), "+v"(vaddr)); // operand addresses are made anew (kept, they spill)
                constexpr int kSlots = C::KK + 4 * C::DT;
                constexpr int kLead = 6;
                constexpr int kCap = CAP ? kSlots / 3 >= 16 ? 16 : kSlots / 3 >= 8 ? 8 : 4 : 0; // slots of the cap,
                constexpr int kSoftmax = kCap + (kSlots >= 24 ? 5 : 2); // of the maximum; 16 half pairs of
                                                                        // probabilities follow
                constexpr int kHalves = 16;
                uint4 ka[C::KK];
                uint2 va[4 * C::DT]; // halves of operand (u, dt)
                const auto read = [&](int i) {
                    if (i < C::KK) {
                        ka[i] = read_k(kat, i);
                    } else if (i < kSlots) {
                        const int x = i - C::KK;
                        va[x] = read_v4(vat, x / (2 * C::DT), x / 2 % C::DT, x & 1);
                    }
                };
#pragma unroll
                for (int i = 0; i < kLead; ++i) {
                    read(i);
                }
                __builtin_amdgcn_sched_barrier(0);
                float tmax = kNegInf;
                float mref = 0.f;
                float sum[2] = {0.f, 0.f};
                float p0 = 0.f;
                float p1 = 0.f;
                uint32_t hp[8];
                uint32_t lp[8];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    next[i] = 0.f;
                }
                unrolled<kSlots>([&](auto slot) {
                    constexpr int i = decltype(slot)::value;
                    read(i + kLead);
                    if constexpr (i < C::KK) {
                        next = mfma_32x32x16<BF16>(ka[i], q[i], next);
                    } else {
                        constexpr int x = i - C::KK;
                        constexpr int u = x / (2 * C::DT);
                        constexpr int dt = x / 2 % C::DT;
                        const uint4 a = make_uint4(va[x & ~1].x, va[x & ~1].y, va[x | 1].x, va[x | 1].y);
                        o[dt] = mfma_32x32x16<BF16>(a, (x & 1) ? pl[j ^ 1][u] : ph[j ^ 1][u], o[dt]);
                    }
#pragma unroll
                    for (int pass = 0; pass < C::NP; ++pass) {
                        if (i == (pass + 1) * kSlots / (C::NP + 1)) {
                            load_pass(j * C::NP + pass, (1 - decltype(bufc)::value) * C::kBuf);
                        }
                    }
                    if constexpr (i < kCap) {
                        constexpr int kPer = 16 / (kCap > 0 ? kCap : 16);
#pragma unroll
                        for (int e = kPer * i; e < kPer * (i + 1); ++e) {
                            const float y = fast_exp2(cap_rate * fabsf(cur[e]));
                            cur[e] = done ? cur[e] : copysignf((1.f - y) * __builtin_amdgcn_rcpf(1.f + y), cur[e]);
                        }
                    } else if constexpr (i < kSoftmax) {
                        // The row maximum and what it changes.
                        constexpr int kPer = 16 / (kSoftmax - kCap - 1);
                        if constexpr (i + 1 < kSoftmax) {
#pragma unroll
                            for (int e = 0; e < kPer; ++e) {
                                tmax = fmaxf(tmax, cur[kPer * (i - kCap) + e]);
                            }
                        } else {
                            tmax = max_halves32(tmax) * mul;
                            raise = tmax > m + kLazyRescaleLog2;
                            const float m_new = raise ? tmax : m;
                            alpha = raise ? fast_exp2(m - m_new) : 1.f;
                            m = m_new;
                            mref = (m == kNegInf ? 0.f : m) - C::kProbLog2Offset;
                        }
                    } else {
                        constexpr int kFrom = (i - kSoftmax) * kHalves / (kSlots - kSoftmax);
                        constexpr int kTo = (i + 1 - kSoftmax) * kHalves / (kSlots - kSoftmax);
                        unrolled<kTo - kFrom>([&](auto half) {
                            constexpr int x = kFrom + decltype(half)::value;
                            constexpr int e = x >> 1;
                            if constexpr ((x & 1) == 0) {
                                p0 = fast_exp2(fmaf(cur[2 * e], mul, -mref));
                                p1 = fast_exp2(fmaf(cur[2 * e + 1], mul, -mref));
                            } else {
                                sum[0] += p0;
                                sum[1] += p1;
                                // The sums come first: the remainder's instruction
                                // overwrites its value.
                                asm("" : "+v"(p0), "+v"(p1) : "v"(sum[0]), "v"(sum[1]));
                                hp[e] = pack2_hw<BF16>(p0, p1);
                                lp[e] = remainder2<BF16>(hp[e], p0, p1, minus_lo, minus_hi);
                                asm volatile("" : "+v"(hp[e]), "+v"(lp[e])); // made here, not where it is used
                            }
                        });
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    ph[j][u] = make_uint4(hp[4 * u], hp[4 * u + 1], hp[4 * u + 2], hp[4 * u + 3]);
                    pl[j][u] = make_uint4(lp[4 * u], lp[4 * u + 1], lp[4 * u + 2], lp[4 * u + 3]);
                }
                l = fmaf(l, alpha, sum[0] + sum[1]);
            };

            // One block of the pipeline: the scores of the next block (K block
            // `j` of the tile's buffers), the product of the last block's
            // probabilities (V block `j`), and between them the softmax of
            // this block, whose tokens start at t.
            // A softcap's kernel caps the scores in the slots, except in blocks
            // that also mask or bias them.
            const auto block = [&](auto jc, auto bufc, int t) {
                f32x16& cur = s[decltype(jc)::value];
                const bool edge = alibi || t < all_lo || t + 32 > all_hi;
                if (edge) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        cur[i] *= scale;
                    }
                    if constexpr (CAP) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            cur[i] = cap * tanh_f32(cur[i] * inv_cap);
                        }
                    }
                    if (alibi) {
                        const float d = static_cast<float>(pos - t - 4 * h);
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            cur[i] -= slope * fabsf(d - static_cast<float>(8 * (i >> 2) + (i & 3)));
                        }
                    }
                    if (t < all_lo || t + 32 > all_hi) {
                        const int from = lo - t - 4 * h;
                        const int upto = hi - t - 4 * h;
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const int tok = 8 * (i >> 2) + (i & 3);
                            cur[i] = tok >= from && tok < upto ? cur[i] : kNegInf;
                        }
                    }
                }
                slots(jc, bufc, edge, edge ? 1.f : CAP ? cap : scale);
                // O holds the products up to the last block's, relative to the old
                // maximum.
                if (__any(raise)) {
#pragma unroll
                    for (int dt = 0; dt < C::DT; ++dt) {
                        o[dt] *= alpha;
                    }
                }
            };

            // Tile k of the pipeline holds the K of blocks 2 k + 1, 2 k + 2 and the V
            // of blocks 2 k - 1, 2 k: the K of block 0 comes ahead of it (through the
            // other buffer), the V of the last block after it.
            if (tiles > 0) {
                const int32_t second_ids = ids;
                ids = first_ids;
                make_addr(t0 - 32); // K block 0, into the other buffer
#pragma unroll
                for (int i = 0; i < C::NP / 2; ++i) {
                    load_pass(i, C::kBuf);
                }
                if constexpr (FP8) {
                    finish_rows(t0 - 32, C::kBuf, 0, C::NP / 2, C::NP);
                }
                ids = second_ids;
                make_addr(t0);
                load_ids(t0 + kTok);
#pragma unroll
                for (int i = 0; i < 2 * C::NP; ++i) {
                    if (i < C::NP || i >= C::NP + C::NP / 2) {
                        load_pass(i, 0);
                    }
                }
                // No block before the first: its V rows are zeros, like its probabilities.
#pragma unroll
                for (int i = 0; i < C::NP / 2; ++i) {
                    *reinterpret_cast<uint4*>(smem + 2 * C::kBuf + (rr + C::RP * i) * D + 8 * cc) =
                        make_uint4(0u, 0u, 0u, 0u);
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    ph[1][u] = make_uint4(0u, 0u, 0u, 0u);
                    pl[1][u] = make_uint4(0u, 0u, 0u, 0u);
                }
                finish_rows(t0, 0, 0, C::NP, C::NP / 2);
                dma_wait();
                __syncthreads();
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    s[0][i] = 0.f;
                }
#pragma unroll
                for (int kk = 0; kk < C::KK; ++kk) {
                    s[0] = mfma_32x32x16<BF16>(read_k(C::kBuf, kk), q[kk], s[0]);
                }
                __syncthreads();
                const auto tile = [&](auto bufc) {
                    make_addr(t0 + kTok);
                    load_ids(t0 + 2 * kTok);
                    block(std::integral_constant<int, 0>{}, bufc, t0);
                    block(std::integral_constant<int, 1>{}, bufc, t0 + 32);
                    finish_rows(t0 + kTok, (1 - decltype(bufc)::value) * C::kBuf, 0, C::NP, 0);
                    dma_wait();
                    __syncthreads();
                    t0 += kTok;
                };
                int k = 0;
                for (; k + 2 <= tiles; k += 2) {
                    tile(std::integral_constant<int, 0>{});
                    tile(std::integral_constant<int, 1>{});
                }
                if (k < tiles) {
                    tile(std::integral_constant<int, 0>{});
                }
                const int last = (2 + (tiles & 1)) * C::kBuf;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
#pragma unroll
                    for (int dt = 0; dt < C::DT; ++dt) {
                        const uint2 v0 = read_v4(last, u, dt, 0);
                        const uint2 v1 = read_v4(last, u, dt, 1);
                        const uint4 a = make_uint4(v0.x, v0.y, v1.x, v1.y);
                        o[dt] = mfma_32x32x16<BF16>(a, ph[1][u], o[dt]);
                        o[dt] = mfma_32x32x16<BF16>(a, pl[1][u], o[dt]);
                    }
                }
                __syncthreads();
            }

            // ---- the segment's rows: the output, or a partial.  They go through
            // the wave's quarter of the LDS, so that whole rows are stored: from the
            // registers an instruction would write 32 bytes of each of 32 rows
            // (5,400 cycles per segment at head_dim 128).
            l = sum_halves32(l);
            const bool whole = empty || (t_lo == 0 && t_hi == span.n);
            const float inv = l > 0.f ? ks.out / l : 0.f;
            if (rows_here > 0) {
                char* const own = reinterpret_cast<char*>(smem) + wave * (C::kBuf * 2);
                int ln = lane; // the places below are made here: kept over the tiles, they spill
                asm volatile("" : "+v"(ln));
                const int n = ln & 31;
                const int h = ln >> 5;
                if (whole) {
                    constexpr int kPlaces = D / 8; // 16-byte chunks per row, at place c ^ row
#pragma unroll
                    for (int dt = 0; dt < C::DT; ++dt) {
#pragma unroll
                        for (int a = 0; a < 4; ++a) {
                            const int dim = (a < 2 ? 0 : C::kSplit) + C::dim0(dt) + 8 * (a & 1);
                            uint2 v;
                            v.x = pack2<BF16>(o[dt][4 * a] * inv, o[dt][4 * a + 1] * inv);
                            v.y = pack2<BF16>(o[dt][4 * a + 2] * inv, o[dt][4 * a + 3] * inv);
                            *reinterpret_cast<uint2*>(own + n * (2 * D) + 16 * ((dim >> 3) ^ (n & (kPlaces - 1))) + 8 * h) = v;
                        }
                    }
                    constexpr int kPer = 64 / kPlaces; // rows per store
                    for (int r0 = 0; r0 < rows_here; r0 += kPer) {
                        const int row = r0 + ln / kPlaces;
                        const int place = ln % kPlaces;
                        const uint4 v = *reinterpret_cast<const uint4*>(own + row * (2 * D) + 16 * place);
                        const int rq = r_first + row;
                        const int i = rq / p.group;
                        if (row < rows_here) {
                            const int64_t at = (static_cast<int64_t>(b) * p.q_len + i) * p.num_heads + kvh * p.group +
                                               (rq - i * p.group);
                            *reinterpret_cast<uint4*>(p.out + at * D + 8 * (place ^ (row & (kPlaces - 1)))) = v;
                        }
                    }
                    if (p.lse != nullptr && h == 0 && live) {
                        store_lse(p.lse, out_row, p.q_len, p.num_heads, m - C::kProbLog2Offset, l);
                    }
                } else {
                    const int64_t row0 = static_cast<int64_t>(2 * w + (t_lo == 0 ? 1 : 0)) * kRows + 32 * wave;
                    constexpr int kPlaces = D / 4;
#pragma unroll
                    for (int dt = 0; dt < C::DT; ++dt) {
#pragma unroll
                        for (int a = 0; a < 4; ++a) {
                            const int dim = (a < 2 ? 0 : C::kSplit) + C::dim0(dt) + 8 * (a & 1) + 4 * h;
                            *reinterpret_cast<float4*>(own + n * (4 * D) + 16 * ((dim >> 2) ^ (n & (kPlaces - 1)))) =
                                make_float4(o[dt][4 * a] * inv, o[dt][4 * a + 1] * inv, o[dt][4 * a + 2] * inv,
                                            o[dt][4 * a + 3] * inv);
                        }
                    }
                    constexpr int kPer = 64 / kPlaces;
#pragma unroll 4
                    for (int r0 = 0; r0 < 32; r0 += kPer) {
                        const int row = r0 + ln / kPlaces;
                        const int place = ln % kPlaces;
                        const float4 v = *reinterpret_cast<const float4*>(own + row * (4 * D) + 16 * place);
                        if (row < rows_here) {
                            *reinterpret_cast<float4*>(p.part_o + (row0 + row) * D + 4 * (place ^ (row & (kPlaces - 1)))) = v;
                        }
                    }
                    if (h == 0 && live) {
                        p.part_lse[row0 + n] = l > 0.f ? (m - C::kProbLog2Offset) + fast_log2(l) : kNegInf;
                    }
                }
            }
            if (!whole && t_lo == 0) {
                // One part more for each share that starts inside the stream.
                int last = w + 1;
                while (last + 1 < workers && share(last + 1) < vs + units - kPrefillSnap) {
                    ++last;
                }
                cut = CutStream{last - w + 1, b, kvh, hg};
            }
            __syncthreads(); // the LDS is free for the next segment
        }
        vs += units;
        if (vs >= x_end) {
            break;
        }
        advance();
    }
    if (tid == 0) {
        cuts[w] = cut;
    }
}

// Merges the cut streams: workgroup (i, w) takes rows R i .. R (i + 1) - 1 of
// the stream whose first part workgroup w of the partition left, if any.  16
// lanes per row; the parts' weights come from their log2-domain LSEs.  W slices
// of the workgroup take every W-th part each and are added through the LDS: a
// long stream cut over the whole chip has hundreds of parts, which one slice
// walks a round trip at a time (512 parts of 2 streams, head_dim 64: the call
// 77 us, with four slices 46).  Bound: the partials' bytes; and the dispatch of
// the workgroups.
template <bool BF16, int D, int R, int W>
__global__ __launch_bounds__(16 * R * W) void prefill_combine_kernel(PartitionParams p) {
    constexpr int E = D / 16; // dims per lane, four at a time: 64 e / 4 + 4 c ..
    const int w = static_cast<int>(blockIdx.y);
    const CutStream cut =
        reinterpret_cast<const CutStream*>(p.part_lse + static_cast<int64_t>(p.tile_workers) * 2 * kRows)[w];
    const int r0 = cut.hg * kRows + static_cast<int>(blockIdx.x) * R;
    if (cut.parts == 0 || r0 >= p.rows) {
        return;
    }
    const int c = threadIdx.x & 15;
    const int slice = static_cast<int>(threadIdx.x) / (16 * R);
    const int r = min(r0 + static_cast<int>(threadIdx.x) / 16 % R, p.rows - 1); // past the rows: the last one again
    const int row = r - cut.hg * kRows;
    const auto slot_row = [&](int k) {
        return static_cast<int64_t>(k == 0 ? 2 * w + 1 : 2 * (w + k)) * kRows + row;
    };
    float mx = kNegInf;
    for (int k = c; k < cut.parts; k += 16) {
        mx = fmaxf(mx, p.part_lse[slot_row(k)]);
    }
    mx = group_max<16>(mx);
    float acc[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        acc[e] = 0.f;
    }
    float sum = 0.f;
    // A part without weight is added too: its row is zeros, or NaN for a query row
    // that holds a NaN (no part of that row has a weight).
#pragma unroll 4
    for (int k = slice; k < cut.parts; k += W) {
        const int64_t at = slot_row(k);
        const float lse = p.part_lse[at];
        const float wt = lse == kNegInf ? 0.f : fast_exp2(lse - mx);
        sum += wt;
        const float* const src = p.part_o + at * D + 4 * c;
        float v[E];
#pragma unroll
        for (int e = 0; e < E; e += 4) {
            *reinterpret_cast<float4*>(v + e) = *reinterpret_cast<const float4*>(src + 16 * e);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            acc[e] = fmaf(wt, v[e], acc[e]);
        }
    }
    if constexpr (W > 1) {
        __shared__ float other[W - 1][E + 1][16 * R];
        const int at = static_cast<int>(threadIdx.x) % (16 * R);
        if (slice > 0) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                other[slice - 1][e][at] = acc[e];
            }
            other[slice - 1][E][at] = sum;
        }
        __syncthreads();
        if (slice > 0) {
            return;
        }
#pragma unroll
        for (int i = 0; i < W - 1; ++i) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                acc[e] += other[i][e][at];
            }
            sum += other[i][E][at];
        }
    }
    const float inv = sum > 0.f ? 1.f / sum : 0.f;
    const int qi = r / p.group;
    const int64_t out_row =
        (static_cast<int64_t>(cut.b) * p.q_len + qi) * p.num_heads + cut.kvh * p.group + (r - qi * p.group);
#pragma unroll
    for (int e = 0; e < E; e += 4) {
        uint2 v;
        v.x = pack2<BF16>(acc[e] * inv, acc[e + 1] * inv);
        v.y = pack2<BF16>(acc[e + 2] * inv, acc[e + 3] * inv);
        *reinterpret_cast<uint2*>(p.out + out_row * D + 4 * c + 16 * e) = v;
    }
    if (p.lse != nullptr && c == 0) {
        store_lse(p.lse, out_row, p.q_len, p.num_heads, mx, sum);
    }
}

template <bool BF16, int D>
hipError_t launch_d(const PartitionParams& p, hipStream_t stream, const LaunchEvents& part_ev,
                    const LaunchEvents& comb_ev) {
    const dim3 grid(p.tile_workers);
    const dim3 block(kThreads);
    if (p.kv_fp8) {
        if (p.softcap_log2 > 0.f) {
            launch_kernel(prefill_kernel<BF16, D, true, true>, grid, block, 0, stream, part_ev, p);
        } else {
            launch_kernel(prefill_kernel<BF16, D, true, false>, grid, block, 0, stream, part_ev, p);
        }
    } else if (p.softcap_log2 > 0.f) {
        launch_kernel(prefill_kernel<BF16, D, false, true>, grid, block, 0, stream, part_ev, p);
    } else {
        launch_kernel(prefill_kernel<BF16, D, false, false>, grid, block, 0, stream, part_ev, p);
    }
    // Few streams of many parts each need the workgroups, and the slices from
    // eight parts a stream on; many cut streams fill the chip as it is, and fewer
    // workgroups are dispatched.  Measured, one slice / four (us, head_dim 128): 32
    // streams (16 parts) 57.5 / 50.2, 128 streams (4 parts) 63.0 / 65.0.
    const int64_t streams = static_cast<int64_t>(p.batch) * p.num_heads_k * p.head_groups;
    if (streams > kComputeUnits / 2) {
        launch_kernel(prefill_combine_kernel<BF16, D, 16, 1>, dim3(kRows / 16, p.tile_workers), dim3(256), 0, stream,
                      comb_ev, p);
    } else if (8 * streams > p.tile_workers) {
        launch_kernel(prefill_combine_kernel<BF16, D, 4, 1>, dim3(kRows / 4, p.tile_workers), dim3(64), 0, stream, comb_ev,
                      p);
    } else {
        launch_kernel(prefill_combine_kernel<BF16, D, 4, 4>, dim3(kRows / 4, p.tile_workers), dim3(256), 0, stream, comb_ev,
                      p);
    }
    return hipGetLastError();
}

} // namespace

hipError_t launch_prefill(const PartitionParams& p, bool bf16, int head_dim, hipStream_t stream,
                          const LaunchEvents& part_ev, const LaunchEvents& comb_ev) {
    switch (head_dim) {
    case 64: return bf16 ? launch_d<true, 64>(p, stream, part_ev, comb_ev) : launch_d<false, 64>(p, stream, part_ev, comb_ev);
    case 128: return bf16 ? launch_d<true, 128>(p, stream, part_ev, comb_ev) : launch_d<false, 128>(p, stream, part_ev, comb_ev);
    case 256: return bf16 ? launch_d<true, 256>(p, stream, part_ev, comb_ev) : launch_d<false, 256>(p, stream, part_ev, comb_ev);
    default: return hipErrorInvalidValue;
    }
}

} // namespace pkv
