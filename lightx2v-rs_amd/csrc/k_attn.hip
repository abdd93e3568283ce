// k_attn.hip -- softmax attention (Backend::attention / causal_attention,
// crates/lightx2v-core/src/backend.rs:276-305; CPU reference
// crates/lightx2v-cpu/src/lib.rs:155-203) on the gfx950 bf16 MFMA.
//
//   out[q, h*d + j] = sum_k softmax_k(q.k / sqrt(d), masked) v[k, j]
//   q [heads, sq, d], k / v [heads, sk, d], mask [sq, sk] (1 = allowed)
//
// k_attn_mfma (d = 64 or 128): one workgroup per (head, 256 queries), eight
// waves of 32 queries, keys in tiles of 64 through LDS, online softmax
// (running max and sum per query, exp2 with log2(e)/sqrt(d) folded in).
// Each wave computes S^T = K Q^T with v_mfma_f32_32x32x16_bf16 (K is the A
// operand, Q the B operand held in registers), so a lane owns one query and
// 32 of its keys: the row max takes one cross-lane step, the row sum one at
// the very end.  P^T stays in the registers it was computed in and is the B
// operand of O^T = V^T P^T; the keys of each 16-key MFMA step are taken in
// the order the S^T layout left them in the lane (4 keys of group g, then 4
// of group g + 2), and V^T's fragments come out of LDS in that same order by
// the transposing read, so neither P nor V is transposed by instructions.
// A per-(query tile, key tile) mask summary skips fully masked tiles and
// reads mask words only in mixed ones.
//
// What bounds it: the matrix cores and the vector ALU of a SIMD together.  A
// 64-key tile is 2 x 1024 cycles of MFMA per SIMD (two waves) and 2 x about
// 155 VALU instructions (32 of them exponentials) that overlap the MFMAs only
// in part.  Dealing MFMAs, LDS reads and softmax out step by step took the
// 12 x 128, 4680 x 6240 frame-causal call from 204 to 152 us (1.45 us per
// tile; with every CU loaded that is 1.4 PFLOP/s, where a plain bf16 matrix
// product of 8192^3 reaches 1.25 here), and 4680 x 18720 over the cache from 600
// to 470.
// Row sums or maxima left out, LDS reads, loads or exponentials left out of
// timing copies: 1 to 8% each; other fragment depths, barrier places and wave
// priorities: within 1%.
//
// k_attn_rows: any d <= 256, one wave per (head, query), keys one at a
// time -- the correctness path for other head sizes.
#include "gemm_common.hpp"
#include "runtime.hpp"

namespace lx2v {

namespace {

constexpr int AQ = 256;  // queries per workgroup (eight waves of 32: K / V tiles shared by 256 queries)
constexpr int AK = 64;   // keys per tile
constexpr int AT = 512;  // threads per workgroup
constexpr int TROW = 2048;  // key tiles whose mask summary is staged in LDS (sk <= 131072)

__device__ __forceinline__ float ld_f(const void *p, size_t i, int dt) {
    return dt == LX2V_DTYPE_BF16 ? bf16_bits_to_f32(((const uint16_t *)p)[i]) : ((const float *)p)[i];
}

// Eight elements i .. i + 7 of an F32 or BF16 array as packed bf16 (RNE).
template <int DT>
__device__ __forceinline__ u32x4 ld8_bf16(const void *p, size_t i) {
    if constexpr (DT == LX2V_DTYPE_BF16) {
        return *(const u32x4 *)((const uint16_t *)p + i);
    } else {
        const f32x4 a = *(const f32x4 *)((const float *)p + i), b = *(const f32x4 *)((const float *)p + i + 4);
        return (u32x4){pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w), pack_bf16x2(b.x, b.y), pack_bf16x2(b.z, b.w)};
    }
}

// Key tiles are staged in LDS as they are, [key][d] rows of bf16: K in a ring
// of three slots, V in two, 16 bytes a lane straight from global memory (f32
// inputs: through registers, rounded).
//
// K: 1 KB blocks, what one wave's load writes: KB rows, 64 bytes of padding
// after each block, and chunk c of row r at chunk c ^ kswz(r) (two bits).  The
// 16 rows a fragment read touches at once then fall in distinct banks (four
// chunk positions x four paddings, or with D = 64 four positions x two half
// rows x two paddings), and a lane's chunk 2 s + hf needs two addresses in
// all (s even, s odd) beside immediates.
//
// V: no padding; 64-byte segment g of row r at segment g ^ vswz(r).  V^T's
// fragments come from the transposing read (ds_read_b64_tr_b16: within each
// 16 lanes, lane 4 j + r gives the address of 4 d of key j and lane i
// receives d i of keys 0..3), whose 32 lanes read 64 bytes of four
// consecutive rows: with the swizzle these are all 64 banks.
template <int D>
struct AttnLds {
    static constexpr int CH = D / 8;            // 16-byte chunks per row
    static constexpr int KB = 64 / CH;          // rows per block
    static constexpr int KBS = 1024 + 64;       // bytes per K block
    static constexpr int KSZ = AK / KB * KBS, VSZ = AK * D * 2;
    static constexpr int V0 = 0, K0 = 2 * VSZ, BYTES = K0 + 3 * KSZ;
    static __device__ __forceinline__ int kswz(int r) { return (r / (KB / 4)) & 3; }
    static __device__ __forceinline__ int vswz(int r) { return (r / (KB / 4)) & (D / 32 - 1); }
};

template <int D, int DT, int ODT>
__global__ __launch_bounds__(AT) void k_attn_mfma(const void *__restrict__ Q, const void *__restrict__ K,
                                                  const void *__restrict__ V, int heads, int sq, int sk, int kvs,
                                                  const uint8_t *__restrict__ tiles, const uint32_t *__restrict__ mbits,
                                                  float c, void *__restrict__ out, uint8_t *__restrict__ omx,
                                                  int omx_rows, float *__restrict__ part, int nsplit) {
    using L = AttnLds<D>;
    constexpr int QS = D / 16;         // 16-wide d steps of S^T
    constexpr int DB = D / 32;         // 32-row d blocks of O^T
    constexpr int KI = AK * D / 8 / AT;  // 16-byte chunks of a K or V tile per thread
    static_assert(KI * AT * 8 == AK * D, "whole rounds");
    __shared__ __attribute__((aligned(16))) uint8_t lds[L::BYTES];

    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, l32 = lane & 31, hf = lane >> 5;
    // XCD-aware order: workgroups b, b + 8, ... run on one XCD, so give each
    // XCD a contiguous range of (head, query tile) items -- the workgroups of
    // a head then share its K / V in one L2.
    //
    // Split mode (nsplit = S > 1, part != null): every item is S pieces, each
    // over about 1/S of its allowed key tiles, writing its unnormalized O^T,
    // running max and sum to `part` for k_attn_merge -- S times the
    // workgroups where the items alone would leave CUs idle.  An XCD's pieces
    // are dispatched from the last query tile down (under a causal mask the
    // tiles that see the most keys start first), an item's S pieces side by
    // side.
    const int nqt = (sq + AQ - 1) / AQ, items = nqt * heads, per_xcd = (items + 7) / 8;
    const bool split = nsplit > 1;
    const int b = blockIdx.x;
    int item = -1, piece = 0;
    if (!split) {
        item = (b % 8) * per_xcd + b / 8;
    } else {
        // XCD x owns positions [lo, hi) of the heads' query tiles, position
        // h nqt + i holding query tile (i st) mod nqt of head h: a stride
        // near nqt / golden ratio, so that the part of a head one XCD gets
        // mixes early and late query tiles (light and heavy under a causal
        // mask) rather than taking a run of them.
        const int lo = (b % 8) * per_xcd, hi = min(items, lo + per_xcd);
        int st = (int)(0.618034f * (float)nqt + 0.5f);
        st = st < 1 ? 1 : st;
        auto gcd = [](int a, int c) {
            while (c) {
                const int t = a % c;
                a = c;
                c = t;
            }
            return a;
        };
        while (gcd(st, nqt) != 1) st++;
        int r0 = nqt, r1 = st % nqt, t0 = 0, t1 = 1;  // extended Euclid: st * sinv = 1 mod nqt
        while (r1) {
            const int qq = r0 / r1, r2 = r0 - qq * r1, t2 = t0 - qq * t1;
            r0 = r1;
            r1 = r2;
            t0 = t1;
            t1 = t2;
        }
        const int sinv = ((t0 % nqt) + nqt) % nqt;
        int r = (b / 8) / nsplit;
        piece = (b / 8) % nsplit;
        for (int t = nqt - 1; t >= 0 && item < 0; t--) {
            // the heads h whose query tile t sits at a position in [lo, hi)
            const int i = (int)(((long long)t * sinv) % nqt);
            const int h0 = lo <= i ? 0 : (lo - i + nqt - 1) / nqt;
            const int h1 = hi - 1 < i ? -1 : (hi - 1 - i) / nqt;
            const int cnt = h1 >= h0 ? h1 - h0 + 1 : 0;
            if (r < cnt)
                item = (h0 + r) * nqt + t;
            else
                r -= cnt;
        }
    }
    if (item < 0 || item >= items) return;
    const int head = item / nqt, qt = item % nqt, nkt = (sk + AK - 1) / AK;
    const int q = qt * AQ + wv * 32 + l32;  // this lane's query
    const bool qin = q < sq;
    const size_t qbase = ((size_t)head * sq + (qin ? q : 0)) * D;
    const size_t kvbase = (size_t)head * kvs * D;  // kvs: rows between heads of K / V (>= sk)

    // Q^T fragments (B operand): d 16 s + 8 hf .. + 8 of this lane's query.
    bf16x8 qf[QS];
#pragma unroll
    for (int s = 0; s < QS; s++)
        qf[s] = __builtin_bit_cast(bf16x8, qin ? ld8_bf16<DT>(Q, qbase + 16 * s + 8 * hf) : (u32x4){});

    // This query tile's key tiles with an allowed pair, in order, as key tile
    // | state << 14 (state 1: every pair allowed, 2: mixed), compacted by
    // wave 0 with ballots.  Without a mask, or past TROW tiles, entry i is
    // tile i itself (all allowed, or read as mixed).
    __shared__ uint16_t list[TROW];
    __shared__ int nlist;
    const bool tlds = tiles && nkt <= TROW;
    if (tlds && wv == 0) {
        int total = 0;
        for (int base = 0; base < nkt; base += 64) {
            const int t = base + lane;
            const int st = t < nkt ? tiles[(size_t)qt * nkt + t] : 0;
            const uint64_t bal = __ballot(st != 0);
            if (st) list[total + __popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)(t | st << 14);
            total += __popcll(bal);
        }
        if (lane == 0) nlist = total;
    }
    if (tlds) __syncthreads();
    const int nall = tlds ? nlist : nkt;
    // This workgroup's entries [i0, i0 + n): all, or in split mode those from
    // the floor(p n / S)-th to the floor((p + 1) n / S)-th (piece p).
    const int i0 = split ? (int)((long long)piece * nall / nsplit) : 0;
    const int n = (split ? (int)((long long)(piece + 1) * nall / nsplit) : nall) - i0;
    const int whole = tiles ? 2 : 1;  // the state of a tile that is not listed
    // key tile | state << 24; -1 past the last
    auto entry = [&](int i) -> int {
        if (i >= n) return -1;
        if (!tlds) return (i0 + i) | whole << 24;
        const int v = list[i0 + i];
        return (v & 0x3FFF) | (v >> 14) << 24;
    };
    auto tile_of = [](int e) { return e & 0xFFFFFF; };
    auto state_of = [](int e) { return e >> 24; };

    f32x16 o[DB];
#pragma unroll
    for (int b = 0; b < DB; b++) o[b] = (f32x16){};
    float m = -INFINITY, lsum = 0.0f;  // running max (log2 domain, scaled); sum over this lane's own keys

    // Global loads through buffer descriptors: keys past sk, and every
    // offset of a tile past the last (kOob), read zero, so the loads need no
    // branch.  K of bf16 inputs goes straight into LDS; f32 K is loaded to
    // registers, rounded and stored at the end of the same iteration.
    constexpr uint32_t ES = DT == LX2V_DTYPE_BF16 ? 2 : 4;
    constexpr int R8 = ES / 2;  // 16-byte loads per 8 elements
    const auto ksrc = make_rsrc((const uint8_t *)K + kvbase * ES, (uint32_t)sk * D * ES);
    const auto vsrc = make_rsrc((const uint8_t *)V + kvbase * ES, (uint32_t)sk * D * ES);
    const uint32_t nw = ((uint32_t)sk + 31) / 32;
    const auto msrc = make_rsrc(mbits, mbits ? (uint32_t)sq * nw * 4 : 0u);
    const uint32_t moff = qin ? (uint32_t)q * nw * 4 : kOob;
    // Round it of a tile: this thread's chunk is row / position of chunk it AT
    // + tid, loaded from the swizzled place.
    uint32_t koff[KI], voff[KI];
#pragma unroll
    for (int it = 0; it < KI; it++) {
        const int ck = it * AT + tid, row = ck / L::CH, pos = ck % L::CH;
        koff[it] = (uint32_t)(row * D + 8 * (pos ^ L::kswz(row))) * ES;
        voff[it] = (uint32_t)(row * D + 8 * (pos ^ (4 * L::vswz(row)))) * ES;
    }
    const uint32_t kdst = __builtin_amdgcn_readfirstlane(lds_addr(lds) + (uint32_t)(L::K0 + wv * L::KBS));
    const uint32_t vdst = __builtin_amdgcn_readfirstlane(lds_addr(lds) + (uint32_t)(L::V0 + wv * 1024));
    // Fragment addresses.  K: chunk (2 s + hf) of row 32 j + l32.  V: for d
    // block b and keys k0 .. k0 + 3, row k0 + j of d 32 b + 16 (group & 1) + 4 r
    // (this lane being 4 j + r of its 16-lane group).
    const uint8_t *const kfr = lds + L::K0 + (l32 / L::KB) * L::KBS + (l32 % L::KB) * (D * 2);
    const uint8_t *const kfr2[2] = {kfr + ((hf ^ L::kswz(l32)) * 16), kfr + (((2 + hf) ^ L::kswz(l32)) * 16)};
    const uint8_t *vfr[DB];
#pragma unroll
    for (int b = 0; b < DB; b++) {
        const int j = (lane / 4) % 4, r = lane % 4, row = 4 * hf + j;
        vfr[b] = lds + L::V0 + row * (D * 2) + ((b ^ L::vswz(row)) * 64) + 32 * ((lane / 16) & 1) + 8 * r;
    }

    u32x4 kr[KI][R8], vr[KI][R8];  // f32 inputs only
    uint32_t mwn[2] = {0u, 0u};    // mask words of the next tile (mixed tiles; kOob reads 0 otherwise)
    // e < 0: past the last tile (the offset's top bit then puts it out of range).
    auto oob = [](bool in) -> uint32_t { return in ? 0u : kOob; };
    auto raw8 = [&](__amdgpu_buffer_rsrc_t r, uint32_t off, u32x4 *d) {
#pragma unroll
        for (int h = 0; h < R8; h++) d[h] = buffer_load_x4(r, off + 16 * h);
    };
    auto bf8 = [&](const u32x4 *d) -> u32x4 {
        const f32x4 a = __builtin_bit_cast(f32x4, d[0]), b = __builtin_bit_cast(f32x4, d[R8 - 1]);
        return (u32x4){pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w), pack_bf16x2(b.x, b.y), pack_bf16x2(b.z, b.w)};
    };
    auto load_k = [&](int it, int slot, int e) {
        const uint32_t off = (koff[it] + (uint32_t)tile_of(e) * (AK * D * ES)) | oob(e >= 0);
        if constexpr (DT == LX2V_DTYPE_BF16)
            dma16_at(ksrc, kdst + slot * L::KSZ + it * (AT / 64) * L::KBS, off);
        else
            raw8(ksrc, off, kr[it]);
    };
    auto load_v = [&](int it, int slot, int e) {
        const uint32_t off = (voff[it] + (uint32_t)tile_of(e) * (AK * D * ES)) | oob(e >= 0);
        if constexpr (DT == LX2V_DTYPE_BF16)
            dma16_at(vsrc, vdst + slot * L::VSZ + it * (AT * 16), off);
        else
            raw8(vsrc, off, vr[it]);
    };
    auto store_k = [&](int it, int slot) {
        if constexpr (DT != LX2V_DTYPE_BF16)
            *(u32x4 *)(lds + L::K0 + slot * L::KSZ + (it * (AT / 64) + wv) * L::KBS + lane * 16) = bf8(kr[it]);
    };
    auto store_v = [&](int it, int slot) {
        if constexpr (DT != LX2V_DTYPE_BF16)
            *(u32x4 *)(lds + L::V0 + slot * L::VSZ + (it * AT + tid) * 16) = bf8(vr[it]);
    };
    auto load_mask = [&](int e) {
        const uint32_t mo = (moff + (uint32_t)tile_of(e) * (AK / 8)) | oob(state_of(e) == 2);
#pragma unroll
        for (int kb = 0; kb < 2; kb++) mwn[kb] = buffer_load_x1(msrc, mo + 4 * kb);
    };
    auto kfrag = [&](const uint8_t *const *kf, int s, int j) {
        return __builtin_bit_cast(bf16x8, *(const u32x4 *)(kf[s & 1] + j * (32 / L::KB) * L::KBS + (s >> 1) * 64));
    };
    // V^T of keys 16 u + 4 hf + 0..3 and 16 u + 8 + 4 hf + 0..3: the 8 keys this
    // lane's P^T registers of step u hold (the order the S^T layout leaves them in).
    auto vfrag = [&](int slot, int u, int b) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s16x4 *lp;
        const uint8_t *const p = vfr[b] + slot * L::VSZ + u * (16 * D * 2);
        const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)p), y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp)(p + 8 * D * 2));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    // Mask a tile's scores in place: a full tile with every pair allowed is
    // left alone; otherwise keys past sk and, in mixed tiles, pairs whose
    // mask bit is clear become -inf.  mwk: the tile's two mask words.
    auto apply_mask = [&](f32x16 *st, int e, const uint32_t *mwk) {
        const int state = state_of(e), k0 = tile_of(e) * AK;
        if (state == 1 && k0 + AK <= sk) return;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            // allowed keys of this 32-key block as bits (mask word, keys
            // before sk), shifted so that register i tests a constant bit
            const int left = sk - (k0 + 32 * j);
            uint32_t allow = state == 2 ? mwk[j] : ~0u;
            allow &= left >= 32 ? ~0u : (left <= 0 ? 0u : (1u << left) - 1u);
            allow >>= 4 * hf;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const bool ok = (allow >> (8 * (i / 4) + (i % 4))) & 1u;
                st[j][i] = ok ? st[j][i] : -INFINITY;
            }
        }
    };

    // One key tile t per iteration:
    //   O^T += V(t-1)^T P(t-1)^T   V(t-1) in V slot P ^ 1 (P = t & 1)
    //   softmax of S(t)            in `cur`, P(t)^T into `pout`
    //   S(t+1) = K(t+1) Q^T        K(t+1) in K slot ks, into `nxt`
    // while V(t+1) is loaded into V slot P ^ 1 and K(t+3) into the K slot that
    // held K(t).  The three are independent, and the code deals them out by hand: a step is one MFMA,
    // the LDS read of the fragment that the MFMA RF - 1 steps on needs, and
    // that step's share of the softmax, fenced so that the order stays.  The
    // matrix cores and the vector ALU of a SIMD then both have work from each
    // of its two waves at any time.
    //
    // One barrier per tile, at the first step of S(t+1): there every wave is past
    // its reads of V(t-1) and K(t), and has V(t) and K(t+2) in LDS (loaded
    // since the barrier before).  Between barriers a wave runs on from one
    // tile into the next with RF - 1 fragments in flight, so no MFMA waits for
    // LDS behind a barrier.
    const float tau = 8.0f;  // rescale O only when a query's max grows by more than 2^8
    constexpr int RF = 4;    // fragment registers (8 measured the same)
    bf16x8 fr[RF];
    uint32_t mw[2] = {0u, 0u};
    int e0 = 0, e1 = 0, e2 = 0, e3 = 0, t = 0, ks = 0;
    auto iter = [&](auto par, auto first, f32x16 *cur, f32x16 *nxt, const u32x4 *pin,
                    u32x4 *pout) __attribute__((always_inline)) {
        constexpr int P = decltype(par)::value;
        constexpr int NPV = decltype(first)::value ? 0 : 4 * DB, NS = 2 * QS, NM = NPV + NS;
        static_assert(NM % RF == 0 && NS > RF && 4 * DB >= RF, "the fragment ring runs on across tiles");
        const uint8_t *const kf[2] = {kfr2[0] + ks * L::KSZ, kfr2[1] + ks * L::KSZ};
        const int kold = ks == 0 ? 2 : ks - 1;  // K(t)'s slot
        // fragment of step I of this tile; past its last step, V(t)'s
        auto fetch = [&](auto i) {
            constexpr int I = decltype(i)::value;
            if constexpr (I < NPV)
                fr[I % RF] = vfrag(P ^ 1, I / DB, I % DB);
            else if constexpr (I < NM)
                fr[I % RF] = kfrag(kf, (I - NPV) / 2, (I - NPV) % 2);
            else
                fr[I % RF] = vfrag(P, (I - NM) / DB, (I - NM) % DB);
        };
        constexpr int SBAR = NPV;  // the barrier's step
        if constexpr (decltype(first)::value) static_for<RF - 1>(fetch);
        const int e4 = entry(t + 4);
        apply_mask(cur, e0, mw);
        __builtin_amdgcn_sched_barrier(0);

        // Softmax of 32 scores: steps S0 .. SR - 1 take the max (from S0 on:
        // the last MFMA of S(t) has then retired), SR the new reference
        // point, the rest exponentials, sums and bf16 pairs.
        constexpr int S0 = 1, SR = S0 + NM / 8, NB = NM - SR - 1;
        auto x = [&](int v) -> float { return cur[v / 16][v % 16]; };
        float tmax = -INFINITY, mn = m, mref = 0.0f, alpha = 1.0f, ps[2] = {0.0f, 0.0f};
        float p[32];
        // (the empty volatile asm statements keep a value's computation in
        // its step: left alone, the compiler sinks it below the branch at the
        // end of the iteration)
        auto sum_pack = [&](int v) {
            ps[v & 1] += p[v];
            asm volatile("" : "+v"(ps[v & 1]));
            if (v & 1) {
                uint32_t w = pack_bf16x2(p[v - 1], p[v]);
                asm volatile("" : "+v"(w));
                pout[v / 8][(v % 8) / 2] = w;
            }
        };
        static_for<NM>([&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (I < NPV) {
                constexpr int u = I / DB, b = I % DB;
                o[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[I % RF], __builtin_bit_cast(bf16x8, pin[u]), o[b], 0, 0, 0);
            } else {
                constexpr int s = (I - NPV) / 2, j = (I - NPV) % 2;
                if constexpr (s == 0) nxt[j] = (f32x16){};
                nxt[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[I % RF], qf[s], nxt[j], 0, 0, 0);
            }
            if constexpr (I == SBAR) {
                if constexpr (DT == LX2V_DTYPE_BF16)
                    wait_vmcnt<0>();
                else
                    wait_vmcnt_lds0<0>();
                asm volatile("s_barrier" ::: "memory");
            }
            fetch(std::integral_constant<int, I + RF - 1>{});
            if constexpr (I == 0) load_mask(e1);
            if constexpr (I > SBAR && I <= SBAR + KI) load_v(I - SBAR - 1, P ^ 1, e1);
            if constexpr (I > SBAR + KI && I <= SBAR + 2 * KI) load_k(I - SBAR - KI - 1, kold, e3);
            if constexpr (I >= S0 && I < SR) {
#pragma unroll
                for (int v = 32 * (I - S0) / (SR - S0); v < 32 * (I - S0 + 1) / (SR - S0); v += 2)
                    tmax = fmaxf(fmaxf(tmax, x(v)), x(v + 1));
            } else if constexpr (I == SR) {
                // The reference point moves only when the tile's max passes it
                // by more than tau: p = 2^(s c - m) <= 2^tau in between, exact
                // in f32, and O is rescaled far less often.  With no key
                // allowed yet (m = -inf) any finite reference works: use 0.
                // The raw v_exp_f32 flushes results below 2^-126 to 0 (no
                // contribution a softmax sum in f32 could register).
                tmax = max_pair32(tmax) * c;
                mn = tmax > m + tau ? tmax : m;
                mref = mn == -INFINITY ? 0.0f : mn;
                alpha = __builtin_amdgcn_exp2f(m - mref);
            } else if constexpr (I > SR) {
                constexpr int B = I - SR - 1, v0 = 32 * B / NB, v1 = 32 * (B + 1) / NB;
#pragma unroll
                for (int v = v0; v < v1; v++) {
                    p[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(x(v), c, -mref));
                    asm volatile("" : "+v"(p[v]));
                    if (v > 0) sum_pack(v - 1);  // (one behind the exponential's latency)
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        sum_pack(31);
#pragma unroll
        for (int it = 0; it < KI; it++) {
            store_v(it, P ^ 1);
            store_k(it, kold);
        }
        lsum = lsum * alpha + (ps[0] + ps[1]);
        m = mn;
        if (__ballot(alpha != 1.0f)) {
            asm volatile("" : "+v"(alpha));  // (the products stay behind the branch: hoisted, every tile pays for them)
#pragma unroll
            for (int b = 0; b < DB; b++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[b][i] *= alpha;
        }
        mw[0] = mwn[0];
        mw[1] = mwn[1];
        e0 = e1;
        e1 = e2;
        e2 = e3;
        e3 = __builtin_amdgcn_readfirstlane(e4);
        t++;
        ks = ks == 2 ? 0 : ks + 1;
    };

    if (n > 0) {
        using std::integral_constant;
        constexpr integral_constant<int, 0> c0{};
        constexpr integral_constant<int, 1> c1{};
        constexpr integral_constant<bool, true> first{};
        constexpr integral_constant<bool, false> later{};
        e0 = __builtin_amdgcn_readfirstlane(entry(0));
        e1 = __builtin_amdgcn_readfirstlane(entry(1));
        e2 = __builtin_amdgcn_readfirstlane(entry(2));
        e3 = __builtin_amdgcn_readfirstlane(entry(3));
        // Tiles 0 .. 2 of K into slots 0 .. 2, V of tile 0, S(0); tile t + 1's K
        // is then in slot (t + 1) % 3 = ks.
        f32x16 sa[2], sb[2];
        u32x4 pa[4], pb[4];
        auto begin = [&](int vslot, f32x16 *cur) __attribute__((always_inline)) {
#pragma unroll
            for (int it = 0; it < KI; it++) {
                load_v(it, vslot, e0);
                store_v(it, vslot);
            }
#pragma unroll
            for (int tl = 0; tl < 3; tl++)
#pragma unroll
                for (int it = 0; it < KI; it++) {
                    load_k(it, tl, tl == 0 ? e0 : (tl == 1 ? e1 : e2));
                    store_k(it, tl);
                }
            load_mask(e0);
            // (Q too: its first use in every iteration would otherwise wait
            // for all loads in flight, the next tile's included)
            wait_vmcnt<0>();
            mw[0] = mwn[0];
            mw[1] = mwn[1];
            __syncthreads();
            cur[0] = cur[1] = (f32x16){};
#pragma unroll
            for (int s = 0; s < QS; s++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    cur[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfrag(kfr2, s, j), qf[s], cur[j], 0, 0, 0);
            ks = 1;
        };
        // Tile 0 takes the V slot that lets the loop below, two tiles a turn,
        // end on slot 0: slot 0 for odd n, slot 1 (and one more tile before
        // the loop) for even n.
        if (n & 1) {
            begin(0, sa);
            iter(c0, first, sa, sb, pb, pa);
        } else {
            begin(1, sb);
            iter(c1, first, sb, sa, pa, pb);
            iter(c0, later, sa, sb, pb, pa);
        }
        while (t < n) {
            iter(c1, later, sb, sa, pa, pb);
            iter(c0, later, sa, sb, pb, pa);
        }
        // the last tile's O^T += V^T P^T, from V slot 0 (its first fragments
        // are in `fr`)
        static_for<4 * DB>([&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (I + RF - 1 < 4 * DB) fr[(I + RF - 1) % RF] = vfrag(0, (I + RF - 1) / DB, (I + RF - 1) % DB);
            o[I % DB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[I % RF], __builtin_bit_cast(bf16x8, pa[I / DB]), o[I % DB], 0, 0, 0);
        });
    }
    {  // the other half of each query's keys
        uint32_t a = __float_as_uint(lsum), b = a;
        swap32(a, b);
        lsum = __uint_as_float(a) + __uint_as_float(b);
    }

    if (!qin) return;
    if (split) {
        // this piece's O^T (unnormalized), running max (log2 domain) and sum
        const size_t slot = (size_t)item * nsplit + piece, row = slot * AQ + (size_t)(q - qt * AQ);
        float *po = part + row * D;
#pragma unroll
        for (int b = 0; b < DB; b++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *(f32x4 *)(po + 32 * b + 8 * g + 4 * hf) =
                    (f32x4){o[b][4 * g], o[b][4 * g + 1], o[b][4 * g + 2], o[b][4 * g + 3]};
        typedef float f32x2_t __attribute__((ext_vector_type(2)));
        if (hf == 0) *(f32x2_t *)(part + (size_t)items * nsplit * AQ * D + row * 2) = (f32x2_t){m, lsum};
        return;
    }
    // No allowed key: 0 / 0 = NaN, as the reference's softmax of all -inf;
    // no key at all (sk = 0): 0, the reference's empty sum.
    const float inv = sk == 0 ? 0.0f : 1.0f / lsum;
    if constexpr (ODT == LX2V_DTYPE_MXE4M3) {
        // MX e4m3 rows of heads * D columns (the input of the O linear): block
        // b of this head is d 32 b .. 32 b + 31, split between lanes l and l
        // + 32 (d 32 b + 8 g + 4 hf + 0..3); the pair's amax gives the block's
        // scale 2^k, codes = RNE e4m3 of v 2^-k (NaN stays NaN: no clamp is
        // needed once |v| 2^-k <= 448), the scale byte goes to the scale
        // array (mx_sidx, omx_rows rows per 128-column group).
        const size_t row0 = (size_t)q * heads * D + (size_t)head * D;
#pragma unroll
        for (int b = 0; b < DB; b++) {
            float v[16];
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                v[i] = o[b][i] * inv;
                amax = fmaxf(amax, fabsf(v[i]));
            }
            amax = fmaxf(amax, __shfl_xor(amax, 32, 64));
            const int k = mx_exponent(amax);
            const float msc = mx_scale(k);
            // lane l ends with the block's codes 0..15, lane l + 32 with 16..31
            uint32_t w[4];
#pragma unroll
            for (int g = 0; g < 4; g++) w[g] = quant4_sc(v + 4 * g, msc);
            swap32(w[0], w[2]);
            swap32(w[1], w[3]);
            *(u32x4 *)((uint8_t *)out + row0 + 32 * b + 16 * hf) = (u32x4){w[0], w[2], w[1], w[3]};
            if (hf == 0) omx[mx_sidx(q, (head * D + 32 * b) / 32, omx_rows)] = (uint8_t)(k + 127);
        }
        return;
    }
    const size_t oi = ((size_t)q * heads + head) * D;
#pragma unroll
    for (int b = 0; b < DB; b++) {
        if constexpr (ODT == LX2V_DTYPE_BF16) {
            // d 8 g + 4 hf .. + 3 in registers 4 g .. + 3: lanes l and l + 32
            // trade halves, lane l storing 8 d of an even g, lane l + 32 of
            // the odd one beside it (32 contiguous bytes of the row)
#pragma unroll
            for (int g = 0; g < 4; g += 2) {
                uint32_t w[4];
#pragma unroll
                for (int h = 0; h < 4; h++) {
                    const int r = 4 * (g + h / 2) + 2 * (h % 2);
                    w[h] = pack_bf16x2(o[b][r] * inv, o[b][r + 1] * inv);
                }
                swap32(w[0], w[2]);
                swap32(w[1], w[3]);
                *(u32x4 *)((uint16_t *)out + oi + 32 * b + 8 * (g + hf)) = (u32x4){w[0], w[1], w[2], w[3]};
            }
        } else {
#pragma unroll
            for (int g = 0; g < 4; g++)
                *(f32x4 *)((float *)out + oi + 32 * b + 8 * g + 4 * hf) =
                    (f32x4){o[b][4 * g] * inv, o[b][4 * g + 1] * inv, o[b][4 * g + 2] * inv, o[b][4 * g + 3] * inv};
        }
    }
}

// Split mode's second pass: the S pieces of each (query, head) row
// combined, O = sum_p O_p 2^(m_p - m) / sum_p l_p 2^(m_p - m) with m = max_p
// m_p, stored as the one-pass kernel stores (F32 / BF16 rows, or MX e4m3 and
// its scale bytes).  A thread per 4 consecutive d of a row, so a 32-d MX
// block is 8 consecutive lanes.
template <int D, int ODT>
__global__ __launch_bounds__(256) void k_attn_merge(const float *__restrict__ part, int nsplit, int heads, int sq,
                                                   int sk, void *__restrict__ out, uint8_t *__restrict__ omx,
                                                   int omx_rows) {
    constexpr int CH = D / 4;
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x, rows = (size_t)sq * heads;
    const bool live = t < rows * CH;
    const size_t r = live ? t / CH : 0;  // q * heads + head, the output row
    const int ch = (int)(t % CH), q = (int)(r / heads), head = (int)(r % heads);
    const int nqt = (sq + AQ - 1) / AQ, qt = q / AQ, items = nqt * heads;
    const size_t row0 = (size_t)(head * nqt + qt) * nsplit * AQ + (size_t)(q - qt * AQ);
    const float *ml = part + (size_t)items * nsplit * AQ * D;
    float mm = -INFINITY;
    for (int p = 0; p < nsplit; p++) mm = fmaxf(mm, ml[2 * (row0 + (size_t)p * AQ)]);
    // an empty piece (m = -inf) weighs 0; no allowed key in any: 0 / 0 = NaN
    float l = 0.0f, v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int p = 0; p < nsplit; p++) {
        const size_t rp = row0 + (size_t)p * AQ;
        const float mp = ml[2 * rp];
        const float w = mp == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mp - mm);
        l = __builtin_fmaf(ml[2 * rp + 1], w, l);
        const f32x4 a = *(const f32x4 *)(part + rp * D + 4 * ch);
        v[0] = __builtin_fmaf(a.x, w, v[0]);
        v[1] = __builtin_fmaf(a.y, w, v[1]);
        v[2] = __builtin_fmaf(a.z, w, v[2]);
        v[3] = __builtin_fmaf(a.w, w, v[3]);
    }
    const float inv = sk == 0 ? 0.0f : 1.0f / l;
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] *= inv;
    const size_t oi = r * D + 4 * ch;
    if constexpr (ODT == LX2V_DTYPE_MXE4M3) {
        float amax = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
        const int k = mx_exponent(amax);
        const float msc = mx_scale(k);
        if (!live) return;
        *(uint32_t *)((uint8_t *)out + oi) = quant4_sc(v, msc);
        if (ch % 8 == 0) omx[mx_sidx(q, (head * D + 4 * ch) / 32, omx_rows)] = (uint8_t)(k + 127);
    } else if constexpr (ODT == LX2V_DTYPE_BF16) {
        if (!live) return;
        typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
        *(u32x2_t *)((uint16_t *)out + oi) = (u32x2_t){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    } else {
        if (!live) return;
        *(f32x4 *)((float *)out + oi) = (f32x4){v[0], v[1], v[2], v[3]};
    }
}

// Any head size d <= 256: one wave per (head, query), lane j owning
// elements j, j + 64, ...; keys one at a time with an online softmax in f32.
__global__ __launch_bounds__(AT) void k_attn_rows(const void *__restrict__ Q, const void *__restrict__ K,
                                                  const void *__restrict__ V, int dt, int heads, int sq, int sk,
                                                  int kvs, int d, const uint8_t *__restrict__ mask, float c,
                                                  void *__restrict__ out, int odt) {
    const int lane = threadIdx.x & 63;
    const size_t row = blockIdx.x * (size_t)(AT / 64) + (threadIdx.x >> 6);  // head * sq + query
    if (row >= (size_t)heads * sq) return;
    const int head = (int)(row / sq), q = (int)(row % sq);
    float qv[4], acc[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int j = lane + 64 * e;
        qv[e] = j < d ? ld_f(Q, row * d + j, dt) : 0.0f;
        acc[e] = 0.0f;
    }
    float m = -INFINITY, lsum = 0.0f;
    for (int key = 0; key < sk; key++) {
        if (mask && !mask[(size_t)q * sk + key]) continue;
        const size_t kb = ((size_t)head * kvs + key) * d;
        float s = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int j = lane + 64 * e;
            if (j < d) s += qv[e] * ld_f(K, kb + j, dt);
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
        const float x = s * c, mn = fmaxf(m, x), alpha = exp2f(m - mn), p = exp2f(x - mn);
        lsum = lsum * alpha + p;
        m = mn;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int j = lane + 64 * e;
            acc[e] = acc[e] * alpha + (j < d ? p * ld_f(V, kb + j, dt) : 0.0f);
        }
    }
    const float inv = sk == 0 ? 0.0f : 1.0f / lsum;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int j = lane + 64 * e;
        if (j >= d) continue;
        const size_t oi = ((size_t)q * heads + head) * d + j;
        if (odt == LX2V_DTYPE_BF16)
            ((uint16_t *)out)[oi] = f32_to_bf16_bits(acc[e] * inv);
        else
            ((float *)out)[oi] = acc[e] * inv;
    }
}

// Mask summary per (256-query, 64-key) tile: 0 no pair allowed, 1 every
// pair allowed, 2 mixed; pairs past sq / sk ignored.  From the packed bits
// (launch_mask_pack's words): a wave per tile reads its 256 queries' two
// words (2 KB, where the bytes would be 16 KB).
__global__ __launch_bounds__(AT) void k_mask_tiles_bits(const uint32_t *__restrict__ bits, int sq, int sk, int nqt,
                                                        int nkt, uint8_t *__restrict__ tiles) {
    const int lane = threadIdx.x & 63, nw = (sk + 31) / 32;
    const size_t t = blockIdx.x * (size_t)(AT / 64) + (threadIdx.x >> 6);
    if (t >= (size_t)nqt * nkt) return;
    const int qt = (int)(t / nkt), kt = (int)(t % nkt);
    bool any = false, all = true;
    for (int i = lane; i < 2 * AQ; i += 64) {
        const int q = qt * AQ + i / 2, j = i % 2, left = sk - (kt * AK + 32 * j);
        if (q >= sq || left <= 0) continue;
        const uint32_t vm = left >= 32 ? ~0u : (1u << left) - 1u;
        const uint32_t w = bits[(size_t)q * nw + 2 * kt + j] & vm;
        any |= w != 0;
        all &= w == vm;
    }
    const bool wany = __ballot(any) != 0, wall = __ballot(!all) == 0;
    if (lane == 0) tiles[t] = !wany ? 0 : (wall ? 1 : 2);
}

// Mask bits: word w of query q holds keys 32 w .. 32 w + 31 (bit = key % 32),
// keys past sk clear.  One wave per (query, 64 keys).
__global__ __launch_bounds__(AT) void k_mask_pack(const uint8_t *__restrict__ mask, int sq, int sk,
                                                  uint32_t *__restrict__ bits) {
    const int lane = threadIdx.x & 63;
    const int nw = (sk + 31) / 32, nw2 = (nw + 1) / 2;
    const size_t t = blockIdx.x * (size_t)(AT / 64) + (threadIdx.x >> 6);
    if (t >= (size_t)sq * nw2) return;
    const int q = (int)(t / nw2), key = (int)(t % nw2) * 64 + lane;
    const bool a = key < sk && mask[(size_t)q * sk + key] != 0;
    const uint64_t b = __ballot(a);
    const int w = key / 32;
    if ((lane & 31) == 0 && w < nw) bits[(size_t)q * nw + w] = (uint32_t)(lane ? b >> 32 : b);
}

// The MemRoPE block mask from temporal indices (dit.rs:643-653): pair
// (q, k) is allowed iff tk[k] <= tq[q].  Bytes: a thread per 4 keys of a
// query row (rows from blockIdx.y); bits: a wave per 64-key block and 64
// queries, one ballot per query; tile summary: a wave per tile from the
// min / max of the tile's query and key indices (all allowed iff
// max tk <= min tq, none iff min tk > max tq).
__global__ __launch_bounds__(AT) void k_mask_temporal_bytes(const uint64_t *__restrict__ tq, const uint64_t *__restrict__ tk,
                                                            int sq, int sk, uint8_t *__restrict__ mask) {
    const int chunks = (sk + 3) / 4;
    for (int q = blockIdx.y; q < sq; q += gridDim.y) {
        const uint64_t tqv = tq[q];
        uint8_t *row = mask + (size_t)q * sk;
        for (int c = blockIdx.x * AT + threadIdx.x; c < chunks; c += gridDim.x * AT) {
            const int k0 = 4 * c;
            uint32_t v = 0;
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (k0 + e < sk && tk[k0 + e] <= tqv) v |= 1u << (8 * e);
            if (k0 + 4 <= sk && (((uintptr_t)(row + k0)) & 3) == 0) {
                *(uint32_t *)(row + k0) = v;
            } else {
                for (int e = 0; e < 4 && k0 + e < sk; e++) row[k0 + e] = (uint8_t)(v >> (8 * e));
            }
        }
    }
}

__global__ __launch_bounds__(AT) void k_mask_temporal_bits(const uint64_t *__restrict__ tq, const uint64_t *__restrict__ tk,
                                                           int sq, int sk, uint32_t *__restrict__ bits) {
    const int lane = threadIdx.x & 63, nw = (sk + 31) / 32, nkb = (sk + 63) / 64;
    const size_t wave = blockIdx.x * (size_t)(AT / 64) + (threadIdx.x >> 6);
    const int kb = (int)(wave % nkb), qg = (int)(wave / nkb);
    if (qg * 64 >= sq) return;
    const int k = 64 * kb + lane;
    const uint64_t tkv = k < sk ? tk[k] : ~0ull;  // keys past sk: never allowed
    const int q1 = min(qg * 64 + 64, sq);
    for (int q = qg * 64; q < q1; q++) {
        const uint64_t b = __ballot(k < sk && tkv <= tq[q]);
        const int w = 2 * kb + (lane >> 5);
        if ((lane & 31) == 0 && w < nw) bits[(size_t)q * nw + w] = (uint32_t)(lane ? b >> 32 : b);
    }
}

__global__ __launch_bounds__(AT) void k_mask_temporal_tiles(const uint64_t *__restrict__ tq, const uint64_t *__restrict__ tk,
                                                            int sq, int sk, int nqt, int nkt, uint8_t *__restrict__ tiles) {
    const int lane = threadIdx.x & 63;
    const size_t t = blockIdx.x * (size_t)(AT / 64) + (threadIdx.x >> 6);
    if (t >= (size_t)nqt * nkt) return;
    const int qt = (int)(t / nkt), kt = (int)(t % nkt);
    uint64_t qmin = ~0ull, qmax = 0, kmin = ~0ull, kmax = 0;
    for (int i = lane; i < AQ; i += 64) {
        const int q = qt * AQ + i;
        if (q < sq) qmin = min(qmin, tq[q]), qmax = max(qmax, tq[q]);
    }
    {
        const int k = kt * AK + lane;
        if (k < sk) kmin = tk[k], kmax = tk[k];
    }
    for (int o = 32; o >= 1; o >>= 1) {
        qmin = min(qmin, (uint64_t)__shfl_xor((unsigned long long)qmin, o, 64));
        qmax = max(qmax, (uint64_t)__shfl_xor((unsigned long long)qmax, o, 64));
        kmin = min(kmin, (uint64_t)__shfl_xor((unsigned long long)kmin, o, 64));
        kmax = max(kmax, (uint64_t)__shfl_xor((unsigned long long)kmax, o, 64));
    }
    if (lane == 0) tiles[t] = kmin > qmax ? 0 : (kmax <= qmin ? 1 : 2);
}

template <int D, int DT>
void attn_mfma_od(hipStream_t s, dim3 grid, const void *q, const void *k, const void *v, int heads, int sq, int sk,
                  int kvs, const uint8_t *tiles, const uint32_t *mask, float c, void *out, int odt, uint8_t *omx,
                  int omx_rows, float *part, int nsplit) {
    if (nsplit > 1) {  // pieces into `part` (the output type only matters to the merge)
        hipLaunchKernelGGL((k_attn_mfma<D, DT, LX2V_DTYPE_F32>), grid, dim3(AT), 0, s, q, k, v, heads, sq, sk, kvs,
                           tiles, mask, c, nullptr, nullptr, 0, part, nsplit);
        const size_t n = (size_t)sq * heads * (D / 4);
        const dim3 mg((unsigned)((n + 255) / 256));
        if (odt == LX2V_DTYPE_BF16)
            hipLaunchKernelGGL((k_attn_merge<D, LX2V_DTYPE_BF16>), mg, dim3(256), 0, s, part, nsplit, heads, sq, sk, out,
                               omx, omx_rows);
        else if (odt == LX2V_DTYPE_MXE4M3)
            hipLaunchKernelGGL((k_attn_merge<D, LX2V_DTYPE_MXE4M3>), mg, dim3(256), 0, s, part, nsplit, heads, sq, sk,
                               out, omx, omx_rows);
        else
            hipLaunchKernelGGL((k_attn_merge<D, LX2V_DTYPE_F32>), mg, dim3(256), 0, s, part, nsplit, heads, sq, sk, out,
                               omx, omx_rows);
        return;
    }
    if (odt == LX2V_DTYPE_BF16)
        hipLaunchKernelGGL((k_attn_mfma<D, DT, LX2V_DTYPE_BF16>), grid, dim3(AT), 0, s, q, k, v, heads, sq, sk, kvs,
                           tiles, mask, c, out, omx, omx_rows, nullptr, 0);
    else if (odt == LX2V_DTYPE_MXE4M3)
        hipLaunchKernelGGL((k_attn_mfma<D, DT, LX2V_DTYPE_MXE4M3>), grid, dim3(AT), 0, s, q, k, v, heads, sq, sk, kvs,
                           tiles, mask, c, out, omx, omx_rows, nullptr, 0);
    else
        hipLaunchKernelGGL((k_attn_mfma<D, DT, LX2V_DTYPE_F32>), grid, dim3(AT), 0, s, q, k, v, heads, sq, sk, kvs,
                           tiles, mask, c, out, omx, omx_rows, nullptr, 0);
}

}  // namespace

bool attention_mfma_supported(size_t d) { return d == 64 || d == 128; }

// Split mode: S = 2, 4 or 8 pieces per (head, query tile), merged in a
// second pass, where the items alone would leave at least half the CUs idle
// (the largest S with items * S <= CUs and 8 S key tiles).  At the Wan
// chunk's 228 items a two-way split balances the causal mask's heavy and
// light query tiles but measured no faster: the merge pass and the piece
// boundaries cost what the balance gains.  LIGHTX2V_HIP_ATTN_SPLIT=0 turns
// it off, =S (2..16) forces S pieces on every MFMA call.
int attention_split(size_t heads, size_t sq, size_t sk, size_t d, int num_cu, size_t *bytes) {
    *bytes = 0;
    if (!attention_mfma_supported(d) || heads == 0 || sq == 0) return 1;
    const char *e = getenv("LIGHTX2V_HIP_ATTN_SPLIT");
    const int mode = e ? atoi(e) : -1;
    const size_t items = ((sq + AQ - 1) / AQ) * heads, nkt = (sk + AK - 1) / AK;
    int S = 1;
    if (mode >= 2)
        S = mode > 16 ? 16 : mode;
    else if (mode != 0)
        while (S < 8 && items * (size_t)S * 2 <= (size_t)num_cu && nkt >= (size_t)S * 16) S *= 2;
    if (S > 1) *bytes = items * (size_t)S * AQ * (d + 2) * 4;
    return S;
}

void launch_mask_tiles_bits(hipStream_t s, const uint32_t *bits, size_t sq, size_t sk, uint8_t *tiles) {
    const int nqt = (int)((sq + AQ - 1) / AQ), nkt = (int)((sk + AK - 1) / AK);
    const size_t n = (size_t)nqt * nkt;
    if (n == 0) return;
    hipLaunchKernelGGL(k_mask_tiles_bits, dim3((unsigned)((n + AT / 64 - 1) / (AT / 64))), dim3(AT), 0, s, bits,
                       (int)sq, (int)sk, nqt, nkt, tiles);
}

void launch_mask_temporal(hipStream_t s, const uint64_t *tq, size_t sq, const uint64_t *tk, size_t sk, uint8_t *mask,
                          uint32_t *bits, uint8_t *tiles) {
    if (sq == 0 || sk == 0) return;
    const size_t chunks = (sk + 3) / 4;
    hipLaunchKernelGGL(k_mask_temporal_bytes,
                       dim3((unsigned)((chunks + AT - 1) / AT), (unsigned)std::min<size_t>(sq, 65535)), dim3(AT), 0, s,
                       tq, tk, (int)sq, (int)sk, mask);
    const size_t waves = ((sk + 63) / 64) * ((sq + 63) / 64);
    hipLaunchKernelGGL(k_mask_temporal_bits, dim3((unsigned)((waves + AT / 64 - 1) / (AT / 64))), dim3(AT), 0, s, tq, tk,
                       (int)sq, (int)sk, bits);
    const int nqt = (int)((sq + AQ - 1) / AQ), nkt = (int)((sk + AK - 1) / AK);
    const size_t n = (size_t)nqt * nkt;
    hipLaunchKernelGGL(k_mask_temporal_tiles, dim3((unsigned)((n + AT / 64 - 1) / (AT / 64))), dim3(AT), 0, s, tq, tk,
                       (int)sq, (int)sk, nqt, nkt, tiles);
}

size_t mask_tile_count(size_t sq, size_t sk) { return ((sq + AQ - 1) / AQ) * ((sk + AK - 1) / AK); }

size_t mask_word_count(size_t sq, size_t sk) { return sq * ((sk + 31) / 32); }

void launch_mask_pack(hipStream_t s, const uint8_t *mask, size_t sq, size_t sk, uint32_t *bits) {
    const size_t n = sq * (((sk + 31) / 32 + 1) / 2);
    if (n == 0) return;
    hipLaunchKernelGGL(k_mask_pack, dim3((unsigned)((n + AT / 64 - 1) / (AT / 64))), dim3(AT), 0, s, mask, (int)sq,
                       (int)sk, bits);
}

void launch_attention(hipStream_t s, const void *q, const void *k, const void *v, int dt, size_t heads, size_t sq,
                      size_t sk, size_t kvs, size_t d, const uint8_t *mask, const uint32_t *mbits,
                      const uint8_t *tiles, void *out, int odt, uint8_t *omx, size_t omx_rows, float *part,
                      int nsplit) {
    if (heads == 0 || sq == 0) return;
    const float c = 1.4426950408889634f / sqrtf((float)d);  // log2(e) / sqrt(d): softmax in base 2
    if (attention_mfma_supported(d)) {
        const size_t items = ((sq + AQ - 1) / AQ) * heads;
        nsplit = part && nsplit > 1 ? nsplit : 1;
        const dim3 grid((unsigned)(8 * nsplit * ((items + 7) / 8)));
        const int hq = (int)heads, iq = (int)sq, ik = (int)sk, is = (int)kvs;
        if (d == 128) {
            if (dt == LX2V_DTYPE_BF16)
                attn_mfma_od<128, LX2V_DTYPE_BF16>(s, grid, q, k, v, hq, iq, ik, is, tiles, mbits, c, out, odt, omx,
                                                   (int)omx_rows, part, nsplit);
            else
                attn_mfma_od<128, LX2V_DTYPE_F32>(s, grid, q, k, v, hq, iq, ik, is, tiles, mbits, c, out, odt, omx,
                                                  (int)omx_rows, part, nsplit);
        } else {
            if (dt == LX2V_DTYPE_BF16)
                attn_mfma_od<64, LX2V_DTYPE_BF16>(s, grid, q, k, v, hq, iq, ik, is, tiles, mbits, c, out, odt, omx,
                                                  (int)omx_rows, part, nsplit);
            else
                attn_mfma_od<64, LX2V_DTYPE_F32>(s, grid, q, k, v, hq, iq, ik, is, tiles, mbits, c, out, odt, omx,
                                                 (int)omx_rows, part, nsplit);
        }
        return;
    }
    const size_t rows = heads * sq;
    hipLaunchKernelGGL(k_attn_rows, dim3((unsigned)((rows + AT / 64 - 1) / (AT / 64))), dim3(AT), 0, s, q, k, v, dt,
                       (int)heads, (int)sq, (int)sk, (int)kvs, (int)d, mask, c, out, odt);
}

}  // namespace lx2v
