// Paged attention for many query rows per kv head (prompts, chunks of prompts) on gfx950.
//
// The kernels of paged_attention.hip give every wave its own K/V stream, which suits a few rows
// per kv head: each K/V byte is read once and memory sets the pace. With hundreds of rows the
// products set it, and there every wave re-reading K/V through L2 and every row group walking the
// whole context (tokens after its last row included) is what costs. Here a workgroup takes 128
// rows of one (sequence, kv head) and its four waves share each K/V tile:
//   * attn_prefill_kernel: a wave owns 32 rows (n = j * group + head-in-group, so GQA heads fill
//     the rows) in the 32 x 32 MFMA layout. A tile of 64 tokens (32 where rows are wider than 256
//     bytes) is copied to LDS straight from the paged cache (buffer_load ... lds) while the tile
//     before is computed; one barrier per tile. S^T = K Q^T puts a query row in one lane pair
//     (l, l + 32), so the softmax needs one cross-lane swap, and its S^T fragment is already the
//     P^T operand of O^T += V^T P^T. bf16 V is read in operand layout by the transposing LDS
//     loads (ds_read_b64_tr_b16).
//   * attn_prefill_plan_kernel: one workgroup lists the work: for each (sequence, row group)
//     its tiles up to the last visible token, in parts of at most the per-workgroup share of the
//     total, ordered longest first, so that the dispatcher's in-order hand-out keeps all CUs busy
//     to the end whatever the lengths.
//   * attn_prefill_combine_kernel: merges the partial states of row groups split into parts.
// Workgroup w takes kv head w % Hkv of list entry w / Hkv: with 8 kv heads the dispatcher's
// round-robin over the 8 XCDs keeps every head's K/V in one XCD's L2. Launches in which no workgroup
// has more than 1024 tokens (f32: 256) to walk, and those of one sequence that fit the chip at once, skip
// the list: the workgroup works its row group and part out from its index. The host bounds the parts
// (prefill_splits in runtime.cpp, from the table's width), the sequence's own context decides them
// (prefill_part_tiles): a table as wide as the longest context a server allows does not make them long.
//
// What bounds it: at head dim 128 a wave's tile of 64 tokens is 32 MFMAs (1024 cycles), about 215
// vector instructions (about 1000 cycles, the exponentials a quarter of them) and 24 KiB of LDS
// reads (192 cycles of the CU's LDS unit, times 8 waves a CU), of which two waves a SIMD overlap a
// part: matrix cores busy 39%, vector units 49% of the time. Without the softmax the same launch
// takes 83% of its time, without the copies 89%. At head dim 64 the vector work sets the pace.
// Measured (us a call with plan and merge, the kernels that stream K/V per wave -> here, on one box):
// four 2048-token prompts, 32/8 heads, head dim 128: 796 -> 183; 300-512 new tokens on contexts of
// 700-8000, 32/8 heads, head dim 64: 341 -> 148; one 64-token chunk on a context of 4096, 32/8 heads:
// 31.7 -> 24.6; four 1024-token prompts, 32/8 heads, head dim 64, f32: 1890 -> 207 (the vector kernel).
// Registers that the workgroups wanted on a CU do not allow (prefill_wgs_per_cu) are spilled, bytes a
// lane: bf16 at head dim 64 8, 96 12, 256 64; f32 at 128 8.
#ifndef KYRO_PREFILL_UNIT
#define KYRO_PREFILL_UNIT 0
#endif
#include "attention_rows.hpp"
#include "common.hpp"
#include "kernels.hpp"

namespace kyro {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kPfThreads = 256;
constexpr int kPfWaves = kPfThreads / 64;
constexpr int kPfBS = 16;  // tokens per slot (slab) of the cache
constexpr int kRawWord3 = 0x00020000;

// Read in place of a missing slab; never written.
__device__ uint4 kPfZeroSlab[kPfBS * 512 / 16];

// Layout of a head dim DR (a multiple of 16) with 2- or 4-byte elements.
template <bool BF16, int DR>
struct PfCfg {
    static constexpr int ES = BF16 ? 2 : 4;
    static constexpr int D = (DR + 31) / 32 * 32;    // columns of V and O held (padded to 32)
    static constexpr int DT = D / 32;                // 32-column tiles of O^T
    static constexpr int KS = DR * ES / 32;          // 32-byte steps of a K or Q row
    static constexpr int CPR = DR * ES / 16;         // 16-byte chunks of a cache row
    static constexpr int NCH = D * ES / 16;          // chunk slots of a row in LDS
    // LDS slab: [NCH / CW column groups][16 tokens][CW chunks]. One copy instruction fills 64
    // consecutive chunks: 4 whole 256-byte rows at CW = 16.
    static constexpr int CW = NCH % 16 == 0 ? 16 : NCH % 8 == 0 ? 8 : 4;
    static constexpr int SLAB = kPfBS * NCH;         // chunks of a slab
    static constexpr int TK = prefill_tile_tokens(BF16, DR);
    static constexpr int NS = TK / kPfBS;            // slabs of a tile
    static constexpr int TT = TK / 32;               // 32-token tiles of S^T
    // f32 head dims where the kernel stands in for the vector kernel, whose sums are trees: short chains
    // of additions (8 in a score, 4 in a tile's O^T += V^T P^T) that are added up in two halves. The error
    // against 64 bits is then level with the vector kernel's over 33 to 4000 tokens (prompts of 200 tokens,
    // head dims 64 / 80 / 96 / 112, 1e-7: 1.15 1.22 1.24 1.23 here, 1.16 1.22 1.26 1.23 there; with two
    // chains per score, as at 128, 1.82 at 112). At head dim 128 two long chains per score and one per
    // output are already closer than the one-block kernel's single chain (1.89 against 2.80).
    static constexpr bool TREE = !BF16 && DR < 128;
    // K rows: chunk c of token t sits in slot c ^ swk(t) of its column group, so that the 16
    // tokens of an operand read (same c) spread over all banks.
    __device__ static constexpr int swk(int t) { return t * CW / 16; }
    // V rows (bf16): the transposing loads of lanes 0..31 take 64 bytes of each of 4 consecutive
    // tokens; slot c ^ swv(t) puts those on distinct banks. f32 V is read 128 bytes of one token
    // at a time: no swizzle.
    __device__ static constexpr int swv(int t) { return BF16 ? 4 * ((t * CW / 16) & (CW / 4 - 1)) : 0; }
    static_assert(DR % 16 == 0 && NCH % 4 == 0, "rows of whole 16-byte chunks");
    static_assert((NS == 4 || NS == 2) && kPfBS * DR * ES <= (int)sizeof(kPfZeroSlab), "tile shape");
};

// Copies one slab (16 tokens of one kv head, `base`) into LDS at dst (wave-uniform). V selects the
// V swizzle. Columns past the head dim (DR < D) repeat the row's last chunk: K's are never read,
// V's reach only output columns that are not stored.
template <class C, bool V, int POL>
__device__ __forceinline__ void copy_slab(uint4* dst, const void* base, int lane) {
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, kPfBS * C::CPR * 16, kRawWord3);
#pragma unroll
    for (int e = 0; e < C::SLAB / 64; ++e) {
        constexpr int kGroup = kPfBS * C::CW;  // chunks of a column group (a multiple of 64)
        const int cg = 64 * e / kGroup;
        const int pos = 64 * e - cg * kGroup + lane;
        const int t = pos / C::CW;
        const int slot = pos % C::CW;
        int c = cg * C::CW + (slot ^ (V ? C::swv(t) : C::swk(t)));
        if (C::CPR < C::NCH) c = min(c, C::CPR - 1);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(dst + 64 * e), 16,
                                                 (t * C::CPR + c) * 16, 0, 0, POL);
    }
}

// A sequence's rows [q0, q0 + q_len) and context length; the bits of what is wrong with them, or 0.
__device__ __forceinline__ int sequence_rows(const AttnArgs& a, int b, int& q0, int& q_len, int& ctx) {
    const int64_t c = a.ctx_lens[b];
    int s0 = b, s1 = b + 1;
    if (a.q_start) {
        s0 = a.q_start[b];
        s1 = a.q_start[b + 1];
    }
    int err = 0;
    if (c < 0 || c > (int64_t)a.max_blocks * a.bs) err |= ERR_CTX_LEN;
    if (s0 < 0 || s1 < s0 || s1 > a.total_q || s1 - s0 > a.max_q_len) err |= ERR_Q_LAYOUT;
    q0 = s0;
    q_len = err ? 0 : s1 - s0;
    ctx = err ? 0 : (int)c;
    return err;
}

// Tiles up to the last token that row group rg of a sequence sees, or -1 where it has no rows.
__device__ __forceinline__ int row_group_tiles(const PrefillArgs& p, int rg, int q_len, int ctx) {
    const int rows = q_len * p.a.group;
    if (rg * kPrefillRows >= rows) return -1;
    const int last = min((rg + 1) * kPrefillRows, rows) - 1;
    const int vis = p.a.causal ? ctx - q_len + last / p.a.group + 1 : ctx;
    return (max(vis, 0) + p.tile_tokens - 1) / p.tile_tokens;
}

// What a wave keeps per row tile.
template <class C>
struct PfState {
    f32x16 o[C::DT];  // O^T: column = the lane's row, rows 32 dt + 8 (i / 4) + 4 h + i % 4
    float m;          // reference the weights are relative to (log2 units, scaled)
    float top;        // running maximum
    float l;          // this lane's share of the row sum
};
// bf16: the reference of a tile's weights is the running maximum, moved up by less than 1 so that it lies
// a whole number above the tile's own maximum: the tile's largest weight is then a power of two, which
// bf16 holds exactly, and no weight passes 1, so that O^T and l stay within the sums of |V| and of ones
// whatever the order of the scores (a reference that may fall 2^30 below it overflows O^T for |V| above
// 1e29; 166.1 against 167.6 us for four 2048-token prompts, head dim 128). Against a reference that lags
// the maximum by up to 2^8 and so hardly ever moves, the rescale of O^T per tile costs 5% of that time
// and lowers the error against 64 bits from 2.09e-3 (2.03e-3 with the plain running maximum) to 1.98e-3,
// where the kernels that stream K/V per wave have 1.97e-3 (contexts of 700-8000 tokens: 2.33e-3,
// 2.23e-3, 2.09e-3, 2.19e-3).

// POL: cache policy of the K/V copies. Streaming where no other row group reads the slabs (a verify
// step's 72 rows per kv head, 64 sequences of 4096 tokens: 201 us with cached loads, 178 us so).
template <bool BF16, int DR, int POL>
__global__ __launch_bounds__(kPfThreads, prefill_wgs_per_cu(BF16, DR)) void attn_prefill_kernel(PrefillArgs p) {
    using C = PfCfg<BF16, DR>;
    const AttnArgs& a = p.a;
    // Two objects per operand: the compiler's waits tell copies into one buffer from reads of
    // the other by the object.
    __shared__ uint4 sK0[C::NS * C::SLAB], sK1[C::NS * C::SLAB];
    __shared__ uint4 sV0[C::NS * C::SLAB], sV1[C::NS * C::SLAB];

    const int entry = (int)blockIdx.x / a.Hkv;
    const int kvh = (int)blockIdx.x - entry * a.Hkv;
    int4 e0, e1;
    if (p.list) {
        if (entry >= p.head[0]) return;
        e0 = p.list[2 * entry];
        e1 = p.list[2 * entry + 1];
    } else {  // no list: row groups from the last one back, each over its parts and all sequences
        const int rest = entry / a.B;
        const int rg = a.row_groups - 1 - rest / p.splits;
        const int s = rest % p.splits;
        e0.x = entry - rest * a.B;
        const int err = sequence_rows(a, e0.x, e0.y, e0.z, e0.w);
        if (err && rest == 0 && kvh == 0 && threadIdx.x == 0) latch_error(a.err, err);
        const int T = row_group_tiles(p, rg, e0.z, e0.w);
        const int len = prefill_part_tiles(p, e0.w);
        if (T < 0 || (s > 0 && s * len >= T)) return;
        e1 = make_int4(rg * kPrefillRows, s * len, min(len, T - s * len),
                       T > len ? (e0.x * a.row_groups + rg) * p.splits + s : -1);
    }
    const int b = __builtin_amdgcn_readfirstlane(e0.x);
    const int q0 = __builtin_amdgcn_readfirstlane(e0.y);
    const int q_len = __builtin_amdgcn_readfirstlane(e0.z);
    const int ctx = __builtin_amdgcn_readfirstlane(e0.w);
    const int row0 = __builtin_amdgcn_readfirstlane(e1.x);
    const int tile0 = __builtin_amdgcn_readfirstlane(e1.y);
    const int nt = __builtin_amdgcn_readfirstlane(e1.z);
    const int part = __builtin_amdgcn_readfirstlane(e1.w);
    SeqInfo si;
    si.b = b;
    si.kvh = kvh;
    si.q0 = q0;
    si.q_len = q_len;
    si.rows = q_len * a.group;
    si.ctx = ctx;

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31;
    const int h = lane >> 5;
    const int wrow0 = row0 + 32 * wave;  // the wave's first row
    const bool active = wrow0 < si.rows;
    const int past = a.causal ? ctx - q_len + 1 : ctx;  // tokens row 0 of the sequence sees
    const int n = wrow0 + col;
    // Rows past the unit take Q = 0 and every token; they are never stored.
    const int vis = n < si.rows ? (a.causal ? past + n / a.group : ctx) : ctx;
    const int wave_lo = a.causal ? past + wrow0 / a.group : ctx;
    const int wave_hi = a.causal ? past + min(wrow0 + 31, si.rows - 1) / a.group : ctx;
    const int wg_hi = a.causal ? past + min(row0 + kPrefillRows - 1, si.rows - 1) / a.group : ctx;
    const int nslots = (max(wg_hi, 0) + kPfBS - 1) / kPfBS;  // slots the row group sees
    const float c = a.scale_log2;

    uint4 q[C::KS];
    {
        const char* qp = reinterpret_cast<const char*>(a.q) + out_row(a, si, n < si.rows ? n : 0) * (C::CPR * 16);
#pragma unroll
        for (int s = 0; s < C::KS; ++s) q[s] = n < si.rows ? load16(qp + (2 * s + h) * 16) : make_uint4(0, 0, 0, 0);
    }

    // Slab ids of the next tiles, one per lane (slab index of kv head 0, -1 for a bad block id):
    // refilled every 64 slots, the following 64 loaded one refill ahead.
    constexpr int kFill = 64 / C::NS;
    auto load_ids = [&](int tile) -> int {
        const int s = tile * C::NS + lane;
        if (s >= nslots) return -1;
        const int blk = s / a.sub;
        const int64_t id = a.table[(size_t)b * a.max_blocks + blk];
        if (id < 0 || id >= a.num_blocks) {
            if (wave == 0) latch_error(a.err, ERR_BLOCK_ID);
            return -1;
        }
        return (int)id * a.Hkv * a.sub + (s - blk * a.sub);
    };
    int ids = load_ids(tile0), ids_next = load_ids(tile0 + kFill);
    uint64_t bad = __ballot(ids < 0);
    auto advance_ids = [&](int i) {  // call once for i = 1, 2, ..
        if (i % kFill == 0) {
            ids = ids_next;
            bad = __ballot(ids < 0);
            ids_next = load_ids(tile0 + i + kFill);
        }
    };
    const size_t slab_bytes = (size_t)kPfBS * C::CPR * 16;
    const size_t head_off = (size_t)kvh * a.bs * (C::CPR * 16);
    auto slab_ptr = [&](const void* cache, int i, int s) -> const void* {
        const int id = __builtin_amdgcn_readlane(ids, (i % kFill) * C::NS + s);
        return id < 0 ? static_cast<const void*>(kPfZeroSlab) : static_cast<const char*>(cache) + id * slab_bytes + head_off;
    };
    // Copies tile i: with four slabs wave w takes slab w of K and of V, with two a whole slab.
    auto issue = [&](int i, uint4* k, uint4* v) {
        if constexpr (C::NS == 4) {
            copy_slab<C, false, POL>(k + wave * C::SLAB, slab_ptr(a.k, i, wave), lane);
            copy_slab<C, true, POL>(v + wave * C::SLAB, slab_ptr(a.v, i, wave), lane);
        } else if (wave < 2) {
            copy_slab<C, false, POL>(k + wave * C::SLAB, slab_ptr(a.k, i, wave), lane);
        } else {
            copy_slab<C, true, POL>(v + (wave - 2) * C::SLAB, slab_ptr(a.v, i, wave - 2), lane);
        }
    };

    // Operand addresses (bytes) of this lane, one per swizzle pattern.
    int kaddr[C::CW / 2];
#pragma unroll
    for (int x = 0; x < C::CW / 2; ++x)
        kaddr[x] = ((lane >> 4) & 1) * (C::SLAB * 16) + (lane & 15) * (C::CW * 16) +
                   ((2 * x + h) ^ C::swk(lane & 15)) * 16;
    const int i16 = lane & 15;
    const int vtok = BF16 ? 4 * h + (i16 >> 2) : 4 * h;
    int vaddr[C::CW / 4];
#pragma unroll
    for (int x = 0; x < C::CW / 4; ++x)
        vaddr[x] = BF16 ? vtok * (C::CW * 16) + ((2 * ((lane >> 4) & 1) + ((i16 & 3) >> 1)) ^ C::swv(vtok) ^ (4 * x)) * 16 +
                              8 * (i16 & 1)
                        : 0;
    const int vaddr32 = vtok * (C::CW * 16) + 4 * col;

    PfState<C> st;
    st.m = st.top = kNegInf;
    st.l = 0.f;
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) st.o[dt][i] = 0.f;

    auto compute = [&](const uint4* kbuf, const uint4* vbuf, int i, uint32_t tbad) {
        const int t0 = (tile0 + i) * C::TK;
        if (!active || t0 >= wave_hi) return;  // nothing visible to this wave (uniform)
        const char* kb = reinterpret_cast<const char*>(kbuf);
        const char* vb = reinterpret_cast<const char*>(vbuf);
        f32x16 S[C::TT];
        constexpr int kGroupBytes = kPfBS * C::CW * 16;
        auto k_operand = [&](int s, int tt) -> uint4 {
            return *reinterpret_cast<const uint4*>(kb + kaddr[s % (C::CW / 2)] + 2 * tt * (C::SLAB * 16) +
                                                   (2 * s / C::CW) * kGroupBytes);
        };
        if constexpr (BF16) {
#pragma unroll
            for (int tt = 0; tt < C::TT; ++tt)
#pragma unroll
                for (int x = 0; x < 16; ++x) S[tt][x] = 0.f;
#pragma unroll
            for (int s = 0; s < C::KS; ++s)
#pragma unroll
                for (int tt = 0; tt < C::TT; ++tt)
                    S[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, k_operand(s, tt)),
                                                                    __builtin_bit_cast(bf16x8, q[s]), S[tt], 0, 0, 0);
            // Keep kAhead operand reads in flight ahead of the products (the compiler's own order
            // waits for each pair; four 1024-token prompts, 16 heads: 60.5 -> 58.3 us). At 256
            // columns the registers do not allow it.
            constexpr int kAhead = DR <= 128 ? (C::KS * C::TT < 8 ? C::KS * C::TT : 8) : DR < 256 ? 4 : 1;
            __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
            for (int x = 0; x < C::KS * C::TT - kAhead; ++x) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x008, kAhead, 0);
        } else {
            static_assert(BF16 || C::TT == 1, "one 32-token tile of scores at a time");
            f32x16 half[2];
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int x = 0; x < 16; ++x) half[y][x] = 0.f;
#pragma unroll
            for (int s = 0; s < C::KS; ++s) {
                const f32x4 kf = __builtin_bit_cast(f32x4, k_operand(s, 0)), qf = __builtin_bit_cast(f32x4, q[s]);
                if constexpr (C::TREE) {
                    f32x16 chain;
#pragma unroll
                    for (int x = 0; x < 16; ++x) chain[x] = 0.f;
#pragma unroll
                    for (int e = 0; e < 4; ++e) chain = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[e], chain, 0, 0, 0);
                    f32x16& to = half[s / (C::KS / 2)];
                    if (s % (C::KS / 2) == 0) to = chain;
                    else to += chain;
                    if (s % 2) __builtin_amdgcn_sched_barrier(0);  // two chains in flight, no more (registers)
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        half[e % 2] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[e], half[e % 2], 0, 0, 0);
                }
            }
            S[0] = half[0] + half[1];
        }
        if (t0 + C::TK > wave_lo || tbad) {
#pragma unroll
            for (int tt = 0; tt < C::TT; ++tt)
#pragma unroll
                for (int x = 0; x < 16; ++x) {
                    const int t = t0 + 32 * tt + 8 * (x / 4) + 4 * h + x % 4;
                    const bool ok = t < vis && !((tbad >> (2 * tt + x / 8)) & 1u);
                    if (!ok) S[tt][x] = kNegInf;
                }
        }
        float mx = S[0][0];
#pragma unroll
        for (int tt = 0; tt < C::TT; ++tt)
#pragma unroll
            for (int x = 0; x < 16; ++x) mx = fmaxf(mx, S[tt][x]);
        {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
            mx = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
        }
        float m_new, alpha;
        if constexpr (BF16) {
            mx *= c;
            st.top = fmaxf(st.top, mx);
            m_new = mx == kNegInf ? st.top : mx + ceilf(st.top - mx);
            // -inf - -inf (nothing visible yet) would be NaN; O^T and l are 0 then.
            alpha = st.m == kNegInf ? 0.f : fast_exp2(st.m - m_new);
        } else {
            // The running maximum, unscaled until the state is stored: a weight's error is relative to
            // its distance from the maximum, and the largest weight is exactly 1.
            m_new = fmaxf(st.m, mx);
            alpha = st.m == kNegInf ? 0.f : fast_exp2((st.m - m_new) * c);
        }
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) st.o[dt] *= alpha;
        st.l *= alpha;
        st.m = m_new;
        const float mref = st.m == kNegInf ? 0.f : st.m;
        float ps = 0.f;
#pragma unroll
        for (int tt = 0; tt < C::TT; ++tt) {
            float pt[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                S[tt][x] = fast_exp2(BF16 ? __builtin_fmaf(S[tt][x], c, -mref) : (S[tt][x] - mref) * c);
                pt[x % 4] += S[tt][x];
            }
            ps += (pt[0] + pt[1]) + (pt[2] + pt[3]);
        }
        st.l += ps;
        // O^T += V^T P^T.
        if constexpr (BF16) {
#pragma unroll
            for (int tt = 0; tt < C::TT; ++tt)
#pragma unroll
                for (int s2 = 0; s2 < 2; ++s2) {
                    uint4 pw;
                    pw.x = pack_bf16x2(S[tt][8 * s2], S[tt][8 * s2 + 1]);
                    pw.y = pack_bf16x2(S[tt][8 * s2 + 2], S[tt][8 * s2 + 3]);
                    pw.z = pack_bf16x2(S[tt][8 * s2 + 4], S[tt][8 * s2 + 5]);
                    pw.w = pack_bf16x2(S[tt][8 * s2 + 6], S[tt][8 * s2 + 7]);
                    const bf16x8 pB = __builtin_bit_cast(bf16x8, pw);
#pragma unroll
                    for (int dt = 0; dt < C::DT; ++dt) {
                        const char* va = vb + vaddr[dt % (C::CW / 4)] + (2 * tt + s2) * (C::SLAB * 16) +
                                         (4 * dt / C::CW) * kGroupBytes;
                        using Ptr = __attribute__((address_space(3))) s16x4*;
                        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Ptr)(va));
                        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Ptr)(va + 8 * C::CW * 16));
                        const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
                        st.o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8, make_uint4(l2.x, l2.y, h2.x, h2.y)), pB, st.o[dt], 0, 0, 0);
                    }
                }
        } else {
            // A tile's products are summed on their own and then added: the chain of additions into O^T
            // is one per tile instead of one per two tokens.
            constexpr int W = C::TREE ? 1 : 2;    // column tiles side by side
            constexpr int NC = C::TREE ? 8 : 1;   // chains of a tile's 16 products
#pragma unroll
            for (int d0 = 0; d0 < C::DT; d0 += W) {
                f32x16 half[2][W];
#pragma unroll
                for (int y = 0; y < NC; ++y) {
                    f32x16 chain[W];
#pragma unroll
                    for (int w = 0; w < W; ++w)
#pragma unroll
                        for (int x = 0; x < 16; ++x) chain[w][x] = 0.f;
#pragma unroll
                    for (int x = y * (16 / NC); x < (y + 1) * (16 / NC); ++x)
#pragma unroll
                        for (int w = 0; w < W; ++w) {
                            const int dt = d0 + w;
                            const float vv = *reinterpret_cast<const float*>(
                                vb + vaddr32 + (x / 8) * (C::SLAB * 16) + (8 * dt / C::CW) * kGroupBytes +
                                (8 * ((x / 4) % 2) + x % 4) * (C::CW * 16) + (8 * dt % C::CW) * 16);
                            chain[w] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, S[0][x], chain[w], 0, 0, 0);
                        }
#pragma unroll
                    for (int w = 0; w < W; ++w) {
                        f32x16& to = half[2 * y / NC][w];
                        if (2 * y % NC == 0) to = chain[w];
                        else to += chain[w];
                    }
                    if (C::TREE && y % 2) __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int w = 0; w < W; ++w) st.o[d0 + w] += C::TREE ? half[0][w] + half[1][w] : half[0][w];
            }
        }
    };

    // The slots of the last block past the context hold anything: V there becomes 0, so that it
    // cannot reach O through a zero probability.
    const int tail_tile = (ctx % kPfBS != 0 && nslots * kPfBS > ctx) ? ctx / C::TK : -1;
    auto landed = [&](int i, uint4* v) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's copies of tile i
        __syncthreads();                     // everyone's; and everyone has left tile i - 1
        if (tile0 + i == tail_tile) {
            const int t0 = ctx % kPfBS, slab = ctx % C::TK / kPfBS;
            for (int x = threadIdx.x; x < (kPfBS - t0) * C::NCH; x += kPfThreads) {
                const int t = t0 + x / C::NCH, pos = x % C::NCH;
                v[slab * C::SLAB + pos / C::CW * (kPfBS * C::CW) + t * C::CW + pos % C::CW] = make_uint4(0, 0, 0, 0);
            }
            __syncthreads();
        }
    };
    auto tile_bad = [&](int i) -> uint32_t { return (uint32_t)(bad >> ((i % kFill) * C::NS)) & ((1u << C::NS) - 1u); };

    if (nt > 0) {
        uint32_t bad_a = tile_bad(0), bad_b = 0;
        issue(0, sK0, sV0);
        for (int i = 0;;) {
            landed(i, sV0);
            if (i + 1 < nt) {
                advance_ids(i + 1);
                bad_b = tile_bad(i + 1);
                issue(i + 1, sK1, sV1);
            }
            compute(sK0, sV0, i, bad_a);
            if (++i >= nt) break;
            landed(i, sV1);
            if (i + 1 < nt) {
                advance_ids(i + 1);
                bad_a = tile_bad(i + 1);
                issue(i + 1, sK0, sV0);
            }
            compute(sK1, sV1, i, bad_b);
            if (++i >= nt) break;
        }
    }

    if (n >= si.rows) return;
    float L = st.l + __shfl_xor(st.l, 32, 64);
    if (part < 0) {
        const float inv = L > 0.f ? 1.f / L : 0.f;
        const size_t row = out_row(a, si, n);
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int d = 32 * dt + 8 * k + 4 * h;
                if (C::D == DR || d < DR)
                    store_row4<DR>(a, row, d, st.o[dt][4 * k] * inv, st.o[dt][4 * k + 1] * inv, st.o[dt][4 * k + 2] * inv,
                                   st.o[dt][4 * k + 3] * inv);
            }
        return;
    }
    // A part's state: m and l by row, O^T in the order the lanes hold it (whole 1 KiB stores).
    const size_t wv = ((size_t)part * a.Hkv + kvh) * kPfWaves + wave;
    if constexpr (!BF16) {
        // Relative to the rounded scaled maximum that the merge weighs parts by.
        const float m = st.m * c;
        const float f = st.m == kNegInf ? 1.f : fast_exp2(__builtin_fmaf(st.m, c, -m));
        st.m = m;
        L *= f;
#pragma unroll
        for (int dt = 0; dt < C::DT; ++dt) st.o[dt] *= f;
    }
    if (h == 0) {
        a.ws_m[wv * 32 + col] = st.m;
        a.ws_l[wv * 32 + col] = L;
    }
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int k = 0; k < 4; ++k)
            reinterpret_cast<float4*>(a.ws_acc)[((wv * C::DT + dt) * 4 + k) * 64 + lane] =
                make_float4(st.o[dt][4 * k], st.o[dt][4 * k + 1], st.o[dt][4 * k + 2], st.o[dt][4 * k + 3]);
}

// Merges the split row groups: a workgroup takes one 32-column tile of one (split row group, kv
// head), a lane the 16 columns of its row that it held in the first pass.
template <int DR>
__global__ __launch_bounds__(kPfThreads) void attn_prefill_combine_kernel(PrefillArgs p) {
    const AttnArgs& a = p.a;
    constexpr int DT = (DR + 31) / 32;
    const int total = (p.list ? p.head[1] : a.B * a.row_groups) * a.Hkv * DT;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int col = lane & 31, h = lane >> 5;
    for (int w = blockIdx.x; w < total; w += gridDim.x) {
        const int dt = w % DT;
        const int x = w / DT;
        const int kvh = x % a.Hkv;
        int4 e, f;  // {q0, q_len, first row, 0}, {first part, parts, 0, 0}
        if (p.list) {
            e = p.comb[2 * (x / a.Hkv)];
            f = p.comb[2 * (x / a.Hkv) + 1];
        } else {
            const int y = x / a.Hkv;
            const int b = y / a.row_groups, rg = y - b * a.row_groups;
            int ctx;
            if (sequence_rows(a, b, e.x, e.y, ctx)) continue;  // the first pass latched it
            const int T = row_group_tiles(p, rg, e.y, ctx);
            const int len = prefill_part_tiles(p, ctx);
            if (T <= len) continue;  // stored by the first pass, or no rows
            e.z = rg * kPrefillRows;
            f.x = y * p.splits;
            f.y = (T + len - 1) / len;
        }
        const int n = e.z + 32 * wave + col;
        if (n >= e.y * a.group) continue;
        const size_t wv0 = ((size_t)f.x * a.Hkv + kvh) * kPfWaves + wave;
        const size_t step = (size_t)a.Hkv * kPfWaves;  // a part's waves to the next part's
        // kBatch parts' loads are issued together (an index past the last part reads the last one
        // again with weight 0), so that a row of few parts costs one memory round trip.
        constexpr int kBatch = 8;
        float M = kNegInf, L = 0.f;
        float4 o[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int i0 = 0; i0 < f.y; i0 += kBatch) {
            float m[kBatch], l[kBatch];
            float4 v[kBatch][4];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const size_t wv = wv0 + min(i0 + i, f.y - 1) * step;
                m[i] = a.ws_m[wv * 32 + col];
                l[i] = a.ws_l[wv * 32 + col];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    v[i][k] = reinterpret_cast<const float4*>(a.ws_acc)[((wv * DT + dt) * 4 + k) * 64 + lane];
            }
            float mb = M;
#pragma unroll
            for (int i = 0; i < kBatch; ++i) mb = fmaxf(mb, m[i]);
            const float mref = mb == kNegInf ? 0.f : mb;
            const float old = fast_exp2(M - mref);
            L *= old;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                o[k].x *= old;
                o[k].y *= old;
                o[k].z *= old;
                o[k].w *= old;
            }
            M = mb;
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const float s = i0 + i < f.y ? fast_exp2(m[i] - mref) : 0.f;
                L += s * l[i];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    o[k].x += s * v[i][k].x;
                    o[k].y += s * v[i][k].y;
                    o[k].z += s * v[i][k].z;
                    o[k].w += s * v[i][k].w;
                }
            }
        }
        const float inv = L > 0.f ? 1.f / L : 0.f;
        SeqInfo si;
        si.q0 = e.x;
        si.kvh = kvh;
        const size_t row = out_row(a, si, n);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int d = 32 * dt + 8 * k + 4 * h;
            if (DR % 32 == 0 || d < DR)
                store_row4<DR>(a, row, d, o[k].x * inv, o[k].y * inv, o[k].z * inv, o[k].w * inv);
        }
    }
}

template <bool BF16, int DR>
void launch_prefill_dim(const PrefillArgs& p, hipStream_t stream) {
    const dim3 grid((unsigned)((long long)p.list_cap * p.a.Hkv));
    if (p.a.stream_kv) attn_prefill_kernel<BF16, DR, kLoadStream><<<grid, kPfThreads, 0, stream>>>(p);
    else attn_prefill_kernel<BF16, DR, kLoadCached><<<grid, kPfThreads, 0, stream>>>(p);
    if (p.part_cap > 0) {
        constexpr long long kMaxGrid = 2048;
        const long long units = (p.list ? (long long)(p.part_cap / 2 + 1) : (long long)p.a.B * p.a.row_groups) * p.a.Hkv *
                                ((DR + 31) / 32);
        attn_prefill_combine_kernel<DR><<<dim3((unsigned)(units < kMaxGrid ? units : kMaxGrid)), kPfThreads, 0, stream>>>(p);
    }
}

#if KYRO_PREFILL_UNIT == 0
// ------------------------------------------------------------------------------------- plan

constexpr int kPlanThreads = 1024;

// Lists the launch's work (head[0] entries, longest first) and the row groups that were split
// (head[1] of them). One workgroup; flat index f is row group f % row_groups of sequence
// f / row_groups (row_groups from the largest q_len).
__global__ __launch_bounds__(kPlanThreads) void attn_prefill_plan_kernel(PrefillArgs p) {
    const AttnArgs& a = p.a;
    constexpr int kBuckets = kPlanThreads;
    __shared__ int bucket[kBuckets];
    __shared__ long long red_sum[kPlanThreads / 64];
    __shared__ int red_max[kPlanThreads / 64];
    __shared__ int wave_tot[kPlanThreads / 64];
    __shared__ int n_parts, n_comb;
    // Up to kPlanThreads sequences are read (and checked) once into LDS.
    __shared__ int s_q0[kPlanThreads], s_ql[kPlanThreads], s_ctx[kPlanThreads];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const bool staged = a.B <= kPlanThreads;
    if (staged) {
        if (t < a.B) {
            const int err = sequence_rows(a, t, s_q0[t], s_ql[t], s_ctx[t]);
            if (err) latch_error(a.err, err);
        }
        bucket[t] = 0;
        if (t == 0) n_parts = n_comb = 0;
        __syncthreads();
    }
    auto tiles = [&](unsigned f, int& b, int& rg, int& q0, int& q_len, int& ctx) -> int {
        b = (int)(f / (unsigned)a.row_groups);
        rg = (int)(f - (unsigned)b * (unsigned)a.row_groups);
        if (staged) {
            q0 = s_q0[b];
            q_len = s_ql[b];
            ctx = s_ctx[b];
        } else {
            const int err = sequence_rows(a, b, q0, q_len, ctx);
            if (err && rg == 0) latch_error(a.err, err);
        }
        return row_group_tiles(p, rg, q_len, ctx);
    };
    const unsigned flat = (unsigned)a.B * (unsigned)a.row_groups;  // below 2^31 (the host checks)
    long long sum = 0;
    int mx = 0;
    int b, rg, q0, q_len, ctx;
    for (unsigned f = t; f < flat; f += kPlanThreads) {
        const int T = tiles(f, b, rg, q0, q_len, ctx);
        sum += max(T, 0);
        mx = max(mx, T);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        sum += __shfl_xor(sum, o, 64);
        mx = max(mx, __shfl_xor(mx, o, 64));
    }
    if (lane == 0) {
        red_sum[wave] = sum;
        red_max[wave] = mx;
    }
    if (!staged) {
        bucket[t] = 0;
        if (t == 0) n_parts = n_comb = 0;
    }
    __syncthreads();
    sum = 0;
    mx = 0;
    for (int w = 0; w < kPlanThreads / 64; ++w) {
        sum += red_sum[w];
        mx = max(mx, red_max[w]);
    }
    // Longest part: a workgroup slot's share of all tiles, and what a part's own cost buys.
    const long long share = (sum * a.Hkv + p.slots - 1) / p.slots + p.split_cost;
    const int C = p.part_cap > 0 ? (int)min((long long)mx, share) : mx;
    auto split = [&](int T, int& len, int& np) {
        len = T;
        np = 1;
        if (T > C) {
            np = (T + C - 1) / C;
            len = (T + np - 1) / np;
            np = (T + len - 1) / len;
        }
    };
    int shift = 0;
    while ((C >> shift) >= kBuckets) ++shift;
    auto bucket_of = [&](int len) { return (C - len) >> shift; };
    for (unsigned f = t; f < flat; f += kPlanThreads) {
        const int T = tiles(f, b, rg, q0, q_len, ctx);
        if (T < 0) continue;
        int len, np;
        split(T, len, np);
        if (np > 1) atomicAdd(&bucket[bucket_of(len)], np - 1);
        atomicAdd(&bucket[bucket_of(T - (np - 1) * len)], 1);
    }
    __syncthreads();
    const int mine = bucket[t];
    const int incl = wave_incl_scan_i(mine);
    if (lane == 63) wave_tot[wave] = incl;
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < kPlanThreads / 64; ++w) {
        before += w < wave ? wave_tot[w] : 0;
        total += wave_tot[w];
    }
    bucket[t] = before + incl - mine;
    __syncthreads();
    for (unsigned f = t; f < flat; f += kPlanThreads) {
        const int T = tiles(f, b, rg, q0, q_len, ctx);
        if (T < 0) continue;
        int len, np;
        split(T, len, np);
        int first = -1;
        if (np > 1) {
            first = atomicAdd(&n_parts, np);
            const int x = atomicAdd(&n_comb, 1);
            if (first + np <= p.part_cap && x < p.part_cap) {
                p.comb[2 * x] = make_int4(q0, q_len, rg * kPrefillRows, 0);
                p.comb[2 * x + 1] = make_int4(first, np, 0, 0);
            }
        }
        for (int i = 0; i < np; ++i) {
            const int nt = i + 1 < np ? len : T - (np - 1) * len;
            const int pos = atomicAdd(&bucket[bucket_of(nt)], 1);
            if (pos < p.list_cap) {
                p.list[2 * pos] = make_int4(b, q0, q_len, ctx);
                p.list[2 * pos + 1] = make_int4(rg * kPrefillRows, i * len, nt, np > 1 ? first + i : -1);
            }
        }
    }
    __syncthreads();
    if (t == 0) {
        // More entries or parts than were sized (a plan/bound mismatch, or row ranges that overlap
        // around an invalid one): latch it and run nothing.
        const bool over = total > p.list_cap || n_parts > p.part_cap;
        if (over) latch_error(a.err, ERR_PLAN);
        p.head[0] = over ? 0 : total;
        p.head[1] = over ? 0 : n_comb;
    }
}
#endif

}  // namespace

#if KYRO_PREFILL_UNIT == 0
hipError_t launch_prefill_wide(const PrefillArgs& p, hipStream_t stream);
hipError_t launch_prefill_f32(const PrefillArgs& p, hipStream_t stream);

hipError_t launch_attention_prefill(const PrefillArgs& p, hipStream_t stream) {
    if (p.list_cap == 0) return hipSuccess;
    if (p.list) attn_prefill_plan_kernel<<<dim3(1), kPlanThreads, 0, stream>>>(p);
    if (!p.a.dtype_bf16) return launch_prefill_f32(p, stream);
    switch (p.a.D) {
        case 64: launch_prefill_dim<true, 64>(p, stream); break;
        case 80: launch_prefill_dim<true, 80>(p, stream); break;
        case 96: launch_prefill_dim<true, 96>(p, stream); break;
        case 112: launch_prefill_dim<true, 112>(p, stream); break;
        case 128: launch_prefill_dim<true, 128>(p, stream); break;
        default: return launch_prefill_wide(p, stream);
    }
    return hipGetLastError();
}
#elif KYRO_PREFILL_UNIT == 1
hipError_t launch_prefill_wide(const PrefillArgs& p, hipStream_t stream) {
    switch (p.a.D) {
        case 160: launch_prefill_dim<true, 160>(p, stream); break;
        case 192: launch_prefill_dim<true, 192>(p, stream); break;
        case 224: launch_prefill_dim<true, 224>(p, stream); break;
        case 256: launch_prefill_dim<true, 256>(p, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
#else
hipError_t launch_prefill_f32(const PrefillArgs& p, hipStream_t stream) {
    switch (p.a.D) {
        case 64: launch_prefill_dim<false, 64>(p, stream); break;
        case 80: launch_prefill_dim<false, 80>(p, stream); break;
        case 96: launch_prefill_dim<false, 96>(p, stream); break;
        case 112: launch_prefill_dim<false, 112>(p, stream); break;
        case 128: launch_prefill_dim<false, 128>(p, stream); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
#endif

}  // namespace kyro
