// gfx950 kernels of the decompress path.
//
//   Huffman decode (decode_withTree/decode, src/huffman.hh:343-372, :679-691)
//   as a chunk-parallel, self-synchronising decode of the archive's single
//   MSB-first bitstream, cut into subsequences of kSubBits bits:
//     k_decode_sync   each thread finds a subsequence's first codeword by
//                     decoding from kLeadBits before it (two decodes of one
//                     stream soon agree, wherever they started), then
//                     decodes the subsequence: start, end and counts.  A
//                     start that is not on the codewords of its predecessor
//                     lists the subsequence
//     k_decode_pass   listed subsequences re-decode from their predecessor's
//                     end; codewords that do not come to the successor's
//                     start list it for the next pass, until no list is left
//     k_decode_tail   the same, passes to the end of a short list in one
//                     workgroup
//     k_decode_sums,  codeword and zero counts per write unit, and their
//     k_decode_scan   prefixes (k_decode_offsets: both for a few units)
//     k_decode_write  final decode from the true starts: quant codes in
//                     16-byte stores + outlier scatter
//                     (src/vecsz_interface.hh:313-317)
//   Lorenzo reconstruction (x_lorenzo_{1,2,3}d1l, src/dualquant.hh:915-1043):
//     k_recon_*       integer segmented scans per Lorenzo block; exact, and
//                     therefore bit-identical to the reference's sequential
//                     fp32 recurrence, whenever every |s| < 2^21 and every
//                     outlier is an integer below 2^21 (all fp32 partial sums
//                     then stay below 2^24); other blocks are listed
//     k_recon_fallback one thread per listed block replays the reference's
//                     fp32 recurrence in its own association
#include "common.hpp"
#include "kernels.hpp"

namespace vsz {

__device__ __forceinline__ uint32_t lane_id2() { return __lane_id(); }

// Pointers with their address space in the type: a pointer that may be either
// LDS or global (or that was loaded from memory) is read by FLAT loads, which
// wait for every global access the wavefront has in flight, its own stores
// among them.
#define VSZ_LDS __attribute__((address_space(3)))
#define VSZ_GLOBAL __attribute__((address_space(1)))
typedef uint32_t U32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t U16x2 __attribute__((ext_vector_type(2)));
using LdsU16 = const VSZ_LDS uint16_t*;
using GlobalU8 = const VSZ_GLOBAL uint8_t*;
using GlobalU16 = const VSZ_GLOBAL uint16_t*;
using GlobalU32 = const VSZ_GLOBAL uint32_t*;
using GlobalU32x4 = const VSZ_GLOBAL U32x4*;

// The bitstream in "aligned space": word w is the big-endian u32 at byte 4w
// of the 16-byte aligned address at or before the stream start; stream bit p
// is aligned-space bit p + shift0.  Bytes before the stream belong to the
// archive header; bytes at or past the stream end are never read and count
// as zero.
struct StreamView {
    GlobalU8 base;
    uint32_t shift0;
    uint64_t nbytes;  // readable bytes from base (through the stream end)

    __device__ __forceinline__ void setup(const uint8_t* stream, uint64_t stream_bits) {
        // pointer arithmetic (not an integer round trip) keeps the global
        // address space visible to the compiler: global_load, not flat_load
        const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(stream) & 15);
        base = (GlobalU8)(stream - mis);
        shift0 = 8 * mis;
        nbytes = mis + stream_bits / 8;
    }
    __device__ __forceinline__ uint32_t word(uint64_t w) const {
        const uint64_t b = 4 * w;
        if (b + 4 <= nbytes) return __builtin_bswap32(((GlobalU32)base)[w]);
        uint32_t v = 0;
        for (int i = 0; i < 4; i++) v = (v << 8) | (b + i < nbytes ? base[b + i] : 0u);
        return v;
    }
};

// Staged words are stored in rows of 17: the 16 words of one subsequence
// followed by a copy of the next row's first word.  Threads of a wavefront,
// each at its own subsequence, then read different LDS banks, and any two
// consecutive words sit side by side (one ds_read2).
constexpr uint32_t kSubWords = kSubBits / 32;
__device__ __forceinline__ uint32_t pad_idx(uint32_t w) { return w + w / kSubWords; }

// 32-bit window whose MSB is bit `lp` of staged words: the words around the
// end of bit lp - 1, so that one alignbit joins them (lp = 0 takes nothing of
// the word before the first, which is only read).
struct PadWin {  // the rows staging above, a copy of word 0 at st[-1]
    const uint32_t* st;
    __device__ __forceinline__ uint32_t operator()(uint32_t lp) const {
        const int32_t t = (int32_t)lp - 1;
        int32_t i = (t >> 5) + (t >> 9);
        asm("" : "+v"(i));  // (else two shifts and two masks for the byte address)
        return __builtin_amdgcn_alignbit(st[i], st[i + 1], ~(uint32_t)t);
    }
};
static_assert(kSubBits == 512, "rows of 16 words");
struct RowWin {  // plain consecutive words
    const uint32_t* row;
    __device__ __forceinline__ uint32_t operator()(uint32_t lp) const {
        const int32_t t = (int32_t)lp - 1, i = t >> 5;
        return __builtin_amdgcn_alignbit(row[i], row[i + 1], ~(uint32_t)t);
    }
};

// The same from global memory, at stream bit p.
struct GlobalWin {
    StreamView sv;
    __device__ __forceinline__ uint64_t operator()(uint64_t p) const {
        const uint64_t a = p + sv.shift0;
        const uint64_t w = a >> 5;
        return ((((uint64_t)sv.word(w)) << 32) | sv.word(w + 1)) << (a & 31);
    }
};

// Whether a list is not empty, or held (every lane of the wavefront calls it).
__device__ __forceinline__ bool listed(const uint32_t* guard) {
    if (!guard) return false;
    const uint32_t lane = min(lane_id2(), kMaxStripes);
    return __any(((GlobalU32)guard)[lane * kCounterWords] != 0);
}
// Whether the field's tables could not be built.
__device__ __forceinline__ bool no_tables(const DecodeArgs& a) { return a.meta && ((GlobalU32)a.meta)[0] != 0; }

// Appends to the list of slot `slot` the lanes with `on` (a subsequence and
// its start), in stripe `stripe`: one counter addition per wavefront.
__device__ __forceinline__ void list_append(const SubState& s, uint32_t pass, uint32_t stripe, bool on, uint64_t j,
                                            uint32_t first) {
    const uint64_t m = __ballot(on);
    if (!m) return;
    const uint32_t lane = lane_id2();
    const int lead = __builtin_ctzll(m);
    uint32_t k = 0;
    if ((int)lane == lead) k = atomicAdd(list_counter(s, pass, stripe), (uint32_t)__popcll(m));
    k = (uint32_t)__builtin_amdgcn_readlane((int)k, lead);
    if (on)
        s.list[pass & 1][stripe * s.stripe_cap + k + __popcll(m & ((1ull << lane) - 1))] = (s.jbase + j) | ((uint64_t)first << 48);
}

// Decode tables as a kernel sees them (T16: the compact ones, Decoder<false>:
// the 32-bit ones).  Decoder yields symbols, CountDecoder counts.
//   look(w)     first-level entry of the codeword (or codewords) at the top of w
//   escape(e)   the codeword is longer than the first level (32-bit tables:
//               or invalid): resolve() walks the deeper tables
//   len, sym    of an entry
//   resolve     e, l <- entry and length of the codeword at lp whose first
//               32 bits (at least 16 of them valid) are w; l = 0: invalid.
//               win is read for the bits past those
template <bool T16>
struct Decoder;

// The deeper compact tables.
struct Deeper16 {
    LdsU16 sub_lds;  // the first n_lds entries
    GlobalU16 sub;   // all of them
    uint32_t n_lds;
    // Entry i.  The empty asm makes a global read's wait part of its own
    // branch: behind the join the wavefronts that read LDS alone would wait
    // too, for all of their stores in flight.
    __device__ __forceinline__ uint32_t entry(uint32_t i) const {
        uint32_t e;
        if (i < n_lds) {
            e = sub_lds[i];
        } else {
            e = sub[i];
            asm volatile("" : "+v"(e));
        }
        return e;
    }
    template <typename W>
    __device__ __forceinline__ void resolve(const W& win, uint32_t w, uint32_t lp, uint32_t& e, uint32_t& l) const {
        e = entry((e << kSubTabBits) | ((w << kLutBits) >> (32 - kSubTabBits)));
        l = e >> 12;
        if (l != 0) {
            l += kLutBits;
            return;
        }
        l = 1;  // (every walk of a full tree ends at a leaf)
        uint32_t used = kLutBits + kSubTabBits;
#pragma unroll 1
        for (int lv = 1; lv < 16; lv++, used += kSubTabBits) {
            e = entry((e << kSubTabBits) | (win(lp + used) >> (32 - kSubTabBits)));
            if (e >> 12) {
                l = used + (e >> 12);
                break;
            }
        }
    }
};

template <>
struct Decoder<true> {
    static constexpr bool kInvalid = false;  // no entry is an invalid path
    const uint16_t* lut;
    Deeper16 deep;
    // The tables are in LDS at lds (TableCopy), n_lds deeper entries of them
    // in a room of a.n_sub16; returns the words they take.
    __device__ __forceinline__ uint32_t attach(const uint32_t* lds, const DecodeArgs& a, uint32_t n_lds) {
        lut = reinterpret_cast<const uint16_t*>(lds);
        deep.sub_lds = (LdsU16)(lut + (1u << kLutBits));
        deep.sub = (GlobalU16)a.tabs + kTabDeep;
        deep.n_lds = n_lds;
        return ((1u << kLutBits) + a.n_sub16) / 2;
    }
    __device__ __forceinline__ uint32_t look(uint32_t w) const {
        uint32_t i = w >> (32 - kLutBits);
        asm("" : "+v"(i));  // (else a shift, a mask and an addition)
        return lut[i];
    }
    static __device__ __forceinline__ bool escape(uint32_t e) { return e < 4096; }
    static __device__ __forceinline__ uint32_t len(uint32_t e) { return e >> 12; }
    static __device__ __forceinline__ uint32_t sym(uint32_t e) { return e & 0xFFF; }
    // Two symbols as the halves of a word.
    static __device__ __forceinline__ uint32_t pack(uint32_t a, uint32_t b) { return (a | (b << 16)) & 0x0FFF0FFFu; }
    template <typename W>
    __device__ __forceinline__ void resolve(const W& win, uint32_t w, uint32_t lp, uint32_t& e, uint32_t& l) const {
        deep.resolve(win, w, lp, e, l);
    }
};

template <>
struct Decoder<false> {
    static constexpr bool kInvalid = true;
    const uint32_t* lut;
    GlobalU32 sub;
    __device__ __forceinline__ uint32_t attach(const uint32_t* lds, const DecodeArgs& a, uint32_t) {
        lut = lds;
        sub = (GlobalU32)a.sub;
        return 1u << kLutBits;
    }
    __device__ __forceinline__ uint32_t look(uint32_t w) const {
        uint32_t i = w >> (32 - kLutBits);
        asm("" : "+v"(i));  // (else a shift, a mask and an addition)
        return lut[i];
    }
    static __device__ __forceinline__ bool escape(uint32_t e) { return (int32_t)e <= 0; }
    static __device__ __forceinline__ uint32_t len(uint32_t e) { return e >> 16; }
    static __device__ __forceinline__ uint32_t sym(uint32_t e) { return e & 0xFFFF; }
    static __device__ __forceinline__ uint32_t pack(uint32_t a, uint32_t b) { return (a & 0xFFFF) | (b << 16); }
    template <typename W>
    __device__ __forceinline__ void resolve(const W& win, uint32_t, uint32_t lp, uint32_t& e, uint32_t& l) const {
        uint32_t used = kLutBits;
#pragma unroll 1
        for (int lv = 0; lv < 16 && (e & kLutSlow); lv++, used += kSubTabBits) {
            e = sub[(e & ~kLutSlow) + (win(lp + used) >> (32 - kSubTabBits))];
            asm volatile("" : "+v"(e));  // (its wait, as in Deeper16::entry)
        }
        l = (e & kLutSlow) ? 0u : (e >> 16) & 0x7F;
    }
};

// The compact counting entry: length << 12 | zeros << 4 | codewords, all the
// whole ones in the 12-bit pattern (3 on average where a codeword has 3 bits);
// zeros are those that decode to symbol 0.
template <bool T16>
struct CountDecoder;
template <>
struct CountDecoder<true> {
    static constexpr bool kInvalid = false;
    static constexpr uint32_t kStep = kLutBits;  // bits of an entry of several codewords, at most
    const uint16_t* lut;
    Deeper16 deep;
    __device__ __forceinline__ uint32_t attach(const uint32_t* lds, const DecodeArgs& a, uint32_t n_lds) {
        lut = reinterpret_cast<const uint16_t*>(lds);
        deep.sub_lds = (LdsU16)(lut + (1u << kLutBits));
        deep.sub = (GlobalU16)a.tabs + kTabDeep;
        deep.n_lds = n_lds;
        return ((1u << kLutBits) + a.n_sub16) / 2;
    }
    __device__ __forceinline__ uint32_t look(uint32_t w) const {
        uint32_t i = w >> (32 - kLutBits);
        asm("" : "+v"(i));  // (else a shift, a mask and an addition)
        return lut[i];
    }
    static __device__ __forceinline__ bool escape(uint32_t e) { return e < 4096; }
    static __device__ __forceinline__ uint32_t len(uint32_t e) { return e >> 12; }
    static __device__ __forceinline__ bool any_zero(uint32_t e0, uint32_t e1) { return ((e0 | e1) & 0xF0) != 0; }
    static __device__ __forceinline__ uint32_t zeros(uint32_t e) { return (e >> 4) & 15; }
    template <typename W>
    __device__ __forceinline__ void resolve(const W& win, uint32_t w, uint32_t lp, uint32_t& e, uint32_t& l) const {
        deep.resolve(win, w, lp, e, l);
        e = (l << 12) | ((e & 0xFFF) == 0 ? 0x11u : 0x01u);
    }
};
template <>
struct CountDecoder<false> : Decoder<false> {
    static constexpr uint32_t kStep = 0;  // single codewords
};

// Copies the tables a kernel keeps in LDS with NT threads: a first level
// (compact: the counting one or the other) and, behind it, as many deeper
// compact entries as there are and fit (n_sub).  fetch() issues every load of
// a thread and put() stores them, so a workgroup can have its tables and its
// bits in flight together and waits for one memory latency; a copy loop of
// one load per round waited for one latency per round, which was most of a
// workgroup's time (the indexed decode of the 512^3 field at 1e-3: 0.28 ->
// 0.16 ms).
template <bool T16, bool COUNT, uint32_t NT>
struct TableCopy {
    static constexpr uint32_t kFirst = (1u << kLutBits) * (T16 ? 2 : 4) / 16;  // vectors of the first level
    static constexpr uint32_t kVecs = (kFirst + (T16 ? kMaxSub16 / 8 : 0) + NT - 1) / NT;
    U32x4 v[kVecs];
    uint32_t n, n_sub;
    __device__ __forceinline__ void fetch(const DecodeArgs& a) {
        n_sub = T16 ? min(a.n_sub16, ((GlobalU32)a.meta)[1]) : 0u;
        n = kFirst + n_sub / 8;
        const GlobalU32x4 first = T16 ? (GlobalU32x4)(a.tabs + (COUNT ? 0u : kTabLut)) : (GlobalU32x4)a.lut;
        const GlobalU32x4 deep = T16 ? (GlobalU32x4)(a.tabs + kTabDeep) : first;
#pragma unroll
        for (uint32_t m = 0; m < kVecs; m++) {
            const uint32_t i = threadIdx.x + m * NT;
            if (i < kFirst)
                v[m] = first[i];
            else if (i < n)
                v[m] = deep[i - kFirst];
        }
    }
    __device__ __forceinline__ void put(uint32_t* lds) const {
#pragma unroll
        for (uint32_t m = 0; m < kVecs; m++)
            if (threadIdx.x + m * NT < n) reinterpret_cast<U32x4*>(lds)[threadIdx.x + m * NT] = v[m];
    }
};

// The two steps from lp on: entries e[], lengths l[] (0: invalid path).  One
// window serves both: its 32 bits hold a codeword of at most 16 bits (or 12
// bits of several) and the first 16 of the next, which is as far as the first
// two table levels look.
template <class D, typename W>
__device__ __forceinline__ void decode_pair(const D& dec, const W& win, uint32_t lp, uint32_t* e, uint32_t* l) {
    const uint32_t w = win(lp);
    e[0] = dec.look(w);
    l[0] = D::len(e[0]);
    uint32_t w2 = w << (l[0] & 31);
    if (D::escape(e[0])) {
        dec.resolve(win, w, lp, e[0], l[0]);
        w2 = l[0] <= 16 ? w << l[0] : win(lp + l[0]);
    }
    e[1] = dec.look(w2);
    l[1] = D::len(e[1]);
    if (D::escape(e[1])) dec.resolve(win, w2, lp + l[0], e[1], l[1]);
}
template <class D, typename W>
__device__ __forceinline__ uint32_t decode_one(const D& dec, const W& win, uint32_t w, uint32_t lp, uint32_t& l) {
    uint32_t e = dec.look(w);
    l = D::len(e);
    if (D::escape(e)) dec.resolve(win, w, lp, e, l);
    return e;
}

// Codewords and zeros (outliers) of the steps that start in [lp, end), added
// to cnt and z; lp ends at the first step's start at or past end, `last` is
// the start of the last round's first step.
// (A step may hold codewords that start past end: they are this
// subsequence's, and the next one starts behind them.)  Returns whether an
// invalid codeword was met (it counts as one of one bit).
//
// Bound by the instructions it issues, so a round is two looks at one window
// and little else (24 vector instructions; 45 and more with the words around
// lp kept in registers, counts taken out of every entry and both looks able to
// walk the deeper tables: the 1 GiB field's sync pass 409 -> 303 us, a 1800 x 3600 slice's 52 -> 40).
// Entries are summed whole: length, zeros and count are the sum's digits, once
// the lengths (lp's own way) and the zeros (rare, summed beside) are taken
// off.  A second look at a longer codeword is dropped; the next round's first
// meets it.
template <class D, typename W>
__device__ __forceinline__ bool decode_count(const D& dec, const W& win, uint32_t& lp, uint32_t end, uint32_t& cnt,
                                             uint32_t& z, uint32_t& last) {
    if constexpr (D::kInvalid) {
        bool bad = false;
        while (lp < end) {
            uint32_t e[2], l[2];
            decode_pair(dec, win, lp, e, l);
            const bool two = lp + max(l[0], 1u) < end;
            bad |= (l[0] == 0) | (two & (l[1] == 0));
            cnt += two ? 2 : 1;
            z += (D::sym(e[0]) == 0) + (two & (D::sym(e[1]) == 0));
            lp += max(l[0], 1u) + (two ? max(l[1], 1u) : 0u);
        }
        return bad;
    } else {
        const uint32_t lp0 = lp, z0 = z;
        uint32_t sum = 0;
        last = lp;
        while (lp < end) {
            const uint32_t w = win(last = lp);
            uint32_t e0 = dec.look(w), l0 = D::len(e0);
            uint32_t e1 = dec.look(w << l0);
            if (D::escape(e0)) {
                dec.resolve(win, w, lp, e0, l0);
                e1 = 0;
            }
            e1 = (!D::escape(e1) & (lp + l0 < end)) ? e1 : 0u;
            sum += e0 + e1;
            lp += l0 + D::len(e1);
            if (__builtin_expect(__any(D::any_zero(e0, e1)), 0)) z += D::zeros(e0) + D::zeros(e1);
        }
        cnt += sum - ((lp - lp0) << 12) - ((z - z0) << 4);
        return false;
    }
}

// The codeword at lp, by the symbols' first level in global memory (a kernel
// that counts keeps the other one in LDS), added to cnt and z.
template <typename W>
__device__ __forceinline__ void count_single(const CountDecoder<true>& dec, const W& win, uint32_t& lp,
                                             const DecodeArgs& a, uint32_t& cnt, uint32_t& z) {
    const uint32_t w = win(lp);
    uint32_t e = ((GlobalU16)a.tabs)[kTabLut + (w >> (32 - kLutBits))], l = e >> 12;
    if (l == 0) dec.deep.resolve(win, w, lp, e, l);
    cnt++;
    z += (e & 0xFFF) == 0;
    lp += l;
}

// Whether the codewords from p on come to bit `to`, and those up to it, added
// to cnt and z.  `to` is a few bits away: one look at the ends of a pattern's
// codewords, mostly (a codeword at a time, each a load, took a re-decode pass
// from 27 to 29 us).
template <typename W>
__device__ __forceinline__ bool count_meet(const CountDecoder<true>& dec, const W& win, uint32_t p, uint32_t to,
                                           const DecodeArgs& a, uint32_t& cnt, uint32_t& z) {
    while (p < to) {
        const uint32_t d = min(to - p, (uint32_t)kLutBits);
        const uint32_t m = ((GlobalU16)a.tabs)[kTabEnds + (win(p) >> (32 - kLutBits))];
        const uint32_t in = m & ((2u << d) - 2);  // ends in the next d bits
        if (to - p <= kLutBits && !(in >> d)) return false;
        if (in == 0 || (m & 1)) {
            // a codeword of more than d bits, or a zero, which has to be found
            count_single(dec, win, p, a, cnt, z);
        } else {
            cnt += __popc(in);
            p += 31 - __clz(in);
        }
    }
    return p == to;
}

// decode_count where the stream may end: behind its end (bit send, at most an
// entry's bits past `end` or more) no codeword counts, so the last steps are
// single codewords.
template <class D, typename W>
__device__ __forceinline__ bool decode_count_to(const D& dec, const W& win, uint32_t& lp, uint32_t end,
                                                uint32_t send, const DecodeArgs& a, uint32_t& cnt, uint32_t& z,
                                                uint32_t& last) {
    if constexpr (D::kStep == 0) {
        return decode_count(dec, win, lp, end, cnt, z, last);
    } else {
        // (a step that starts below lim ends at or before the stream's end)
        const uint32_t lim = min(end, send > D::kStep ? send - (D::kStep - 1) : 0u);
        const bool bad = decode_count(dec, win, lp, lim, cnt, z, last);
        while (lp < end) count_single(dec, win, lp, a, cnt, z);  // (never, where lim is end)
        return bad;
    }
}

// Whether either half of w is 0 after taking the halves' minima with those of
// more words (pk_min).
__device__ __forceinline__ uint32_t pk_min(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(U16x2, a), __builtin_bit_cast(U16x2, b)));
}
__device__ __forceinline__ bool pk_has_zero(uint32_t w) { return ((w & 0xFFFFu) == 0) | ((w >> 16) == 0); }

// Stages aligned-space words from w0 (a multiple of 4) with NT threads, at
// most VECS 16-byte vectors each: fetch() issues every load, the put()s store
// (see TableCopy).  Vectors past the stream's readable bytes are zero, the
// one that holds its end is read word by word.
template <uint32_t VECS, uint32_t NT>
struct StageCopy {
    U32x4 v[VECS];
    __device__ __forceinline__ void fetch(const StreamView& sv, uint64_t w0, uint32_t nvec) {
        const GlobalU32x4 src = (GlobalU32x4)sv.base + w0 / 4;
        // whole vectors from w0 on, of those wanted
        const uint64_t whole = sv.nbytes / 16 > w0 / 4 ? sv.nbytes / 16 - w0 / 4 : 0;
        const uint32_t lim = (uint32_t)min<uint64_t>(whole, nvec);
#pragma unroll
        for (uint32_t m = 0; m < VECS; m++) {
            v[m] = U32x4{0, 0, 0, 0};
            if (threadIdx.x + m * NT < lim) v[m] = src[threadIdx.x + m * NT];
        }
#pragma unroll
        for (uint32_t m = 0; m < VECS; m++)
            v[m] = U32x4{__builtin_bswap32(v[m].x), __builtin_bswap32(v[m].y), __builtin_bswap32(v[m].z),
                         __builtin_bswap32(v[m].w)};
        if (lim < nvec && (sv.nbytes & 15)) {
#pragma unroll
            for (uint32_t m = 0; m < VECS; m++) {
                if (threadIdx.x + m * NT == lim) {
                    const uint64_t w = w0 + 4 * lim;
                    v[m] = U32x4{sv.word(w), sv.word(w + 1), sv.word(w + 2), sv.word(w + 3)};
                }
            }
        }
    }
    // Into rows (pad_idx), the first nw words; st[-1] is written too.
    __device__ __forceinline__ void put_rows(uint32_t* st, uint32_t nw) const {
#pragma unroll
        for (uint32_t m = 0; m < VECS; m++) {
            const uint32_t k = 4 * (threadIdx.x + m * NT);
            if (k < nw) {
                // four consecutive words never straddle a row
                uint32_t* d = st + pad_idx(k);
                d[0] = v[m].x;
                d[1] = v[m].y;
                d[2] = v[m].z;
                d[3] = v[m].w;
                if (k % kSubWords == 0) d[-1] = v[m].x;  // the previous row's copy of its successor (word 0's: PadWin)
            }
        }
    }
    // Into consecutive words (16-byte aligned).
    __device__ __forceinline__ void put(uint32_t* st, uint32_t nvec) const {
#pragma unroll
        for (uint32_t m = 0; m < VECS; m++)
            if (threadIdx.x + m * NT < nvec) reinterpret_cast<U32x4*>(st)[threadIdx.x + m * NT] = v[m];
    }
};

constexpr uint32_t kSyncWg = 512;             // subsequences decoded per workgroup
constexpr uint32_t kSyncStride = kSyncWg - 1;  // ... whose results it writes (the first one's belong to the workgroup before)
// Bits decoded before a subsequence to find its first codeword.
constexpr uint32_t kLeadBits = 288;
static_assert(kLeadBits <= kSubBits, "the lead lies in one row");
// A row for the first subsequence's lead, and the tail its last codewords'
// windows read: the last starts before bit kSubBits + shift0 (<= 120) of its
// row, the second of its pair up to 64 bits later, and a decode reads at most
// 72 + 64 bits on (the deepest table walk of an invalid path, words read ahead).
constexpr uint32_t kSyncStageWords = (kSyncWg + 1) * kSubWords + 12;
constexpr uint32_t kSyncStageLds = kSyncStageWords + kSyncStageWords / kSubWords + 1;
constexpr int kManyWrong = 16;  // of a wavefront's starts (see decode_sync_unit)
constexpr uint32_t kSyncLdsWords = 1 + kSyncStageLds + kSyncWg;  // dynamic LDS after the tables

// Workgroup `unit` of the sync pass: subsequences unit * kSyncStride on.
template <bool T16>
__device__ __forceinline__ void decode_sync_unit(const DecodeArgs& a, const SubState& s, DecSummary* sum,
                                                 uint64_t unit, uint32_t stripe) {
    extern __shared__ __align__(16) uint32_t lds[];
    if (no_tables(a)) return;  // (the whole workgroup)
    CountDecoder<T16> dec;
    uint32_t* st;
    StreamView sv;
    sv.setup(a.stream, a.stream_bits);
    const uint64_t J0 = unit * kSyncStride;
    // the stage starts one row before subsequence J0 (but not before the stream)
    const uint64_t Jst = J0 ? J0 - 1 : 0;
    {
        TableCopy<T16, true, kSyncWg> tc;
        StageCopy<(kSyncStageWords + 4 * kSyncWg - 1) / (4 * kSyncWg), kSyncWg> sc;
        tc.fetch(a);
        sc.fetch(sv, Jst * kSubWords, (kSyncStageWords + 3) / 4);
        st = lds + dec.attach(lds, a, tc.n_sub) + 1;
        tc.put(lds);
        sc.put_rows(st, kSyncStageWords);
    }
    uint32_t* own_e = st + kSyncStageLds;
    lds_sync();
    const uint32_t t = threadIdx.x;
    const uint64_t j = J0 + t;
    const bool live = j < a.nsub;
    bool bad = false;
    // stage bits: the subsequence's first bit, its first codeword, its target
    const uint32_t s0 = (uint32_t)(j - Jst) * kSubBits + sv.shift0;
    uint32_t first = s0, e0 = s0, cnt = 0, z = 0, lp = s0, last;
    if (live) {
        const PadWin win{st};
        const uint64_t left = a.stream_bits - j * kSubBits;
        e0 += (uint32_t)min<uint64_t>(kSubBits, left);
        const uint32_t send = s0 + (uint32_t)min<uint64_t>(2 * kSubBits, left);
        if (j) {
            lp = s0 - kLeadBits;
            uint32_t lc = 0, lz = 0;
            (void)decode_count_to(dec, win, lp, s0, send, a, lc, lz, last);  // (an invalid path here is a wrong start's)
            first = lp;
        }  // (the stream starts with a codeword)
        bad = decode_count_to(dec, win, lp, e0, send, a, cnt, z, last);
        own_e[t] = lp;
    }
    lds_sync();
    bool wrong = false;
    uint32_t pred = s0;
    if (live && (t > 0 || j == 0)) {
        if (t > 0) pred = own_e[t - 1];
        wrong = t > 0 && pred != first;
        if constexpr (T16) {
            // The lead and the subsequence before each stopped behind a step,
            // of several codewords maybe: up to 11 bits past s0 and, in
            // general, not at the same codeword.  A start on the codewords of
            // the other is right all the same, and only the ones in between
            // change hands.  (Compared as they are, subsequences in a run of
            // one short codeword, a constant stretch of a field, never settle:
            // with 2^21 noise values and 2^21 of one 2-bit codeword every
            // start of the run was listed in each of 8,190 passes, 92 ms a
            // call where it is 0.16 now.)  Only where it is so for many of a
            // wavefront, as in a run: the five or six of other fields, mostly
            // on other codewords indeed, can as well be listed, and looking at
            // them in every wavefront took the 1 GiB field's sync pass from
            // 304 to 308 us.
            const uint32_t to = max(pred, first);
            if (__popcll(__ballot(wrong)) >= kManyWrong && wrong && to <= e0) {
                uint32_t n = 0, nz = 0;
                if (count_meet(dec, PadWin{st}, min(pred, first), to, a, n, nz)) {
                    cnt += first > pred ? n : 0u - n;
                    z += first > pred ? nz : 0u - nz;
                    first = pred;
                    wrong = false;
                }
            }
        }
        s.b[j] = (uint8_t)(first - s0);
        s.e[j] = (uint8_t)(lp - e0);
        s.cz[j] = cnt | (z << 16);
        if (bad && !wrong) atomicOr(&sum->error, 1u);
    }
    list_append(s, 0, stripe, wrong, j, pred - s0);
}

template <bool T16>
__global__ void __launch_bounds__(kSyncWg) k_decode_sync(DecodeArgs a, SubState s, DecSummary* sum) {
    decode_sync_unit<T16>(a, s, sum, blockIdx.x, blockIdx.x % s.nstripe);
}

// Re-decode pass: each listed subsequence j is decoded from its listed start
// (the true end of j - 1); this gives its start, counts and end.  An end other
// than the one j + 1's data was computed from lists j + 1, from that end, for
// the next pass.  Chains shorten by at least one per pass.  Workgroups take
// 256 entries at a time, one per thread; a thread stages its entry's row (the
// subsequence plus the tail its last codeword may read) in LDS with
// independent 16-byte loads, all in flight together, then decodes it.
//
// A row is aligned-space words 16 j .. 16 j + kRowWords - 1, 16-byte aligned
// like the stream base: the last codeword starts before local bit 512 +
// shift0 (<= 632), the second of its pair up to 64 bits later, and a decode
// reads at most 72 + 64 bits on (see kSyncStageWords), so the last word read
// is word 25.
constexpr uint32_t kRowWords = 28;    // seven 16-byte loads
constexpr uint32_t kRowStride = 29;   // odd: the lanes' reads of one word index fall in different banks
constexpr uint32_t kPassGrid = 1024;  // persistent workgroups of a pass (at most ~4 resident per CU)
__device__ __forceinline__ void stage_row(uint32_t* __restrict__ row, const StreamView& sv, uint64_t j) {
    const uint64_t w0 = j * kSubWords;
    if (4 * (w0 + kRowWords) <= sv.nbytes) {
        const GlobalU32x4 src = (GlobalU32x4)sv.base + w0 / 4;
        U32x4 v[kRowWords / 4];
#pragma unroll
        for (uint32_t m = 0; m < kRowWords / 4; m++) v[m] = src[m];
#pragma unroll
        for (uint32_t m = 0; m < kRowWords / 4; m++) {
            row[4 * m] = __builtin_bswap32(v[m].x);
            row[4 * m + 1] = __builtin_bswap32(v[m].y);
            row[4 * m + 2] = __builtin_bswap32(v[m].z);
            row[4 * m + 3] = __builtin_bswap32(v[m].w);
        }
    } else {  // the stream's last rows: bytes past its end read as zero
        for (uint32_t w = 0; w < kRowWords; w++) row[w] = sv.word(w0 + w);
    }
}
// Entry `ent` (jbase taken off its number) of pass `pass`'s list, in the
// thread's own LDS row.  Returns whether j + 1 (set) is to be listed, from
// over bits past its first.
template <bool T16>
__device__ __forceinline__ bool redecode_entry(const DecodeArgs& a, const SubState& s, const CountDecoder<T16>& dec,
                                               uint32_t* row, uint64_t ent, DecSummary* sum, uint64_t& next,
                                               uint32_t& over) {
    const uint64_t j = (ent & ((1ull << 48) - 1)) - s.jbase;
    const uint32_t first = (uint32_t)(ent >> 48);
    StreamView sv;
    sv.setup(a.stream, a.stream_bits);
    stage_row(row, sv, j);  // the thread's own row: no barrier
    const RowWin win{row};
    const uint64_t left = a.stream_bits - j * kSubBits;
    const uint32_t tl = (uint32_t)min<uint64_t>(kSubBits, left) + sv.shift0;
    const uint32_t send = (uint32_t)min<uint64_t>(2 * kSubBits, left) + sv.shift0;
    uint32_t lp = first + sv.shift0, cnt = 0, z = 0;
    const uint32_t old = s.e[j], to = tl + old;
    next = j + 1;
    uint32_t last = lp;
    if (decode_count_to(dec, win, lp, tl, send, a, cnt, z, last)) atomicOr(&sum->error, 1u);
    if constexpr (T16) {
        // Another end than j + 1 starts from, which does as well if these
        // codewords come to it (see decode_sync_unit): they are j's up to it.
        if (lp != to && to <= send) {
            uint32_t n = 0, nz = 0;
            if (count_meet(dec, win, lp < to ? lp : last, to, a, n, nz)) {
                if (lp < to) {
                    cnt += n, z += nz;
                } else {
                    n = nz = 0;
                    (void)count_meet(dec, win, to, lp, a, n, nz);
                    cnt -= n, z -= nz;
                }
                lp = to;
            }
        }
    }
    over = lp - tl;
    s.b[j] = (uint8_t)first;
    s.cz[j] = cnt | (z << 16);
    if (over == old) return false;
    s.e[j] = (uint8_t)over;
    return next < a.nsub;
}

// A pass over stripe `stripe` by workgroups b of nb.  (Whole wavefronts go
// round together: list_append.)
template <bool T16>
__device__ __forceinline__ void decode_pass_stripe(const DecodeArgs& a, const SubState& s, uint32_t pass, DecSummary* sum,
                                                   uint32_t stripe, uint32_t b, uint32_t nb) {
    const uint32_t m = *list_counter(s, pass, stripe);
    if (b == 0 && threadIdx.x == 0) *list_counter(s, pass + 2, stripe) = 0;  // the list after next
    if ((uint64_t)b * 256 >= m) return;                                      // whole workgroup
    extern __shared__ __align__(16) uint32_t lds[];
    CountDecoder<T16> dec;
    uint32_t* rows;
    {
        TableCopy<T16, true, 256> tc;
        tc.fetch(a);
        rows = lds + dec.attach(lds, a, tc.n_sub);
        tc.put(lds);
    }
    lds_sync();  // the tables
    for (uint64_t e0 = b * 256ull + (threadIdx.x & ~63u); e0 < m; e0 += nb * 256ull) {
        const uint64_t e = e0 + lane_id2();
        bool on = false;
        uint64_t next = 0;
        uint32_t over = 0;
        if (e < m)
            on = redecode_entry<T16>(a, s, dec, rows + threadIdx.x * kRowStride,
                                     s.list[pass & 1][stripe * s.stripe_cap + e], sum, next, over);
        list_append(s, pass + 1, stripe, on, next, over);
    }
}

// Workgroup b takes entries of stripe b % nstripe.
template <bool T16>
__global__ void __launch_bounds__(256) k_decode_pass(DecodeArgs a, SubState s, uint32_t pass, DecSummary* sum) {
    decode_pass_stripe<T16>(a, s, pass, sum, blockIdx.x % s.nstripe, blockIdx.x / s.nstripe, gridDim.x / s.nstripe);
}

// The end of a redo that a few chains of wrong starts make long: one
// workgroup resolves pass `pass`'s list in place, all passes' worth, when it
// holds at most kTailWg entries (else it does nothing).  A pass over such a
// list is latency: about 4 us of launch and tables around 5 to 13 of work, and
// a host check with its launches every so many passes (a walk of 2^26 values,
// 24 passes: decompress 933 us with passes alone, 770 with the last 16 of them
// in here).
// Rounds are passes as k_decode_pass makes them, with the lists in LDS and a
// barrier between them that also orders the subsequences' state.  Bounded:
// what is left after kTailRounds goes back to the list.
constexpr uint32_t kTailWg = kTailList;  // an entry per thread
constexpr uint32_t kTailRounds = 512;
template <bool T16>
__global__ void __launch_bounds__(kTailWg) k_decode_tail(DecodeArgs a, SubState s, uint32_t pass, DecSummary* sum) {
    extern __shared__ __align__(16) uint32_t lds[];
    if (no_tables(a)) return;
    const uint32_t t = threadIdx.x;
    // entry t of the stripes one after the other (nstripe <= 32: a lane each)
    const uint32_t k = lane_id2() < s.nstripe ? min(*list_counter(s, pass, lane_id2()), 2 * kTailWg) : 0u;
    const uint32_t ends = wave_scan_dpp(k);
    uint32_t m = lane63(ends);
    if (m == 0 || m > kTailWg) return;  // (the whole workgroup)
    uint64_t at = 0;
    for (uint32_t q = 0; q < s.nstripe; q++) {
        const uint32_t q1 = (uint32_t)__builtin_amdgcn_readlane((int)ends, (int)q);
        const uint32_t q0 = q1 - (uint32_t)__builtin_amdgcn_readlane((int)k, (int)q);
        if (t >= q0 && t < q1) at = q * s.stripe_cap + (t - q0);
    }
    uint64_t* list = s.list[pass & 1];
    CountDecoder<T16> dec;
    uint32_t* p = lds;
    {
        TableCopy<T16, true, kTailWg> tc;
        tc.fetch(a);
        p += dec.attach(lds, a, tc.n_sub);
        tc.put(lds);
    }
    uint32_t* rows = p;
    uint64_t* ents = reinterpret_cast<uint64_t*>(rows + kTailWg * kRowStride);  // two lists, by turns
    uint32_t* n_ents = reinterpret_cast<uint32_t*>(ents + 2 * kTailWg);         // their counters
    if (t < 2) n_ents[t] = 0;
    uint64_t ent = t < m ? list[at] : 0;
    mem_sync();
    uint32_t cur = 0;
    for (uint32_t r = 0; m && r < kTailRounds; r++, cur ^= 1) {
        if (t < m) {
            uint64_t next = 0;
            uint32_t over = 0;
            if (redecode_entry<T16>(a, s, dec, rows + t * kRowStride, ent, sum, next, over))
                ents[cur * kTailWg + atomicAdd(n_ents + cur, 1u)] = (s.jbase + next) | ((uint64_t)over << 48);
        }
        mem_sync();
        m = n_ents[cur];
        ent = t < m ? ents[cur * kTailWg + t] : 0;
        if (t == 0) n_ents[cur ^ 1] = 0;  // the next round's
        mem_sync();
    }
    if (t < m) list[t] = ent;
    if (t < s.nstripe) *list_counter(s, pass, t) = t == 0 ? m : 0u;
}

__device__ __forceinline__ float read_f32_bytes(const uint8_t* p) {
    uint32_t v = (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
    return __uint_as_float(v);
}

// The stream span of workgroup w's segments [256 w, 256 w + 256) in the
// indexed decode: from the first segment's first codeword to the next
// workgroup's (the stream end for the last), as aligned-space words w_lo ..
// w_lo + nwords (plus kIdxSpanPad words the last codewords' windows read).
// fits: the span is staged in LDS by k_decode_indexed_staged (a span that
// runs backwards, from a damaged index, never fits).
constexpr uint32_t kIdxSpanWords = 9984;  // stage capacity: ~9.75 bits per symbol over 256 segments
constexpr uint32_t kIdxSpanPad = 6;
constexpr uint32_t kIdxSpanOver = 264;    // a damaged stream: 128 codewords of up to 64 bits past the span, and the windows past those
struct IdxSpan {
    uint64_t bs, be;  // stream bits of the span
    uint64_t w_lo, nwords;
    bool fits;
};
__device__ __forceinline__ IdxSpan idx_span(const uint64_t* __restrict__ index, const IdxLayout& L,
                                            uint64_t total_bits, const StreamView& sv, uint64_t w) {
    const uint64_t* grp = index + L.grp;
    const uint32_t* rel_bits = reinterpret_cast<const uint32_t*>(index + L.rel_bits);
    const uint64_t g0 = w * 256, g1 = min<uint64_t>(g0 + 256, L.nseg);
    const uint64_t bs = grp[2 * (g0 / kIdxGroup)] + rel_bits[g0];
    const uint64_t be = g1 < L.nseg ? grp[2 * (g1 / kIdxGroup)] + rel_bits[g1] : total_bits;
    IdxSpan sp;
    sp.bs = bs;
    sp.be = be;
    sp.w_lo = (bs + sv.shift0) >> 7 << 2;  // (16-byte aligned)
    sp.nwords = be >= bs ? ((be + sv.shift0) >> 5) - sp.w_lo + kIdxSpanPad : 0;
    sp.fits = be >= bs && sp.nwords <= kIdxSpanWords;
    return sp;
}

// Window over the stream for the indexed decode: 64 bits held in a register
// (relative bit b0 at its MSB, refilled a word at a time by the caller);
// windows beyond it (the deeper levels of codewords over 32 bits) are read
// from memory.  Relative bit 0 is aligned-space bit 32 * w0.
struct CursorWin {
    StreamView sv;
    uint64_t w0;
    uint64_t buf;
    uint32_t b0;
    __device__ __forceinline__ uint32_t operator()(uint32_t lp) const {
        const uint32_t o = lp - b0;
        if (o <= 32) return (uint32_t)((buf << o) >> 32);
        const uint64_t ab = 32 * w0 + lp;
        const uint64_t wi = ab >> 5;
        return __builtin_elementwise_fshl(sv.word(wi), sv.word(wi + 1), (uint32_t)(ab & 31));
    }
};

// Decode with a decode index, for the workgroups whose span does not fit the
// LDS stage of k_decode_indexed_staged (it returns at once for the others):
// thread g decodes segment g (kIdxSeg symbols)
// from the segment's first codeword, reading the stream through a 64-bit
// register window refilled from 16-byte groups loaded ahead, so no LDS
// staging of the bits and no synchronisation is needed.  Codes leave through
// LDS: every lane puts 32 symbols (four 16-byte units) in its wavefront's
// stage, then the wavefront writes the stage so that each store instruction
// covers 16 whole 64-byte pieces instead of 64 scattered 16-byte units.
// Outliers are written from the segment's outlier rank on.  A segment that
// does not end where the next one starts (an index that does not belong to
// this stream) is an error.
constexpr uint32_t kIdxFlush = 32;                       // symbols per lane between stage flushes
constexpr uint32_t kIdxLaneWords = 16 + 1;               // u32 per lane in the stage (odd: no bank conflicts)
constexpr uint32_t kIdxStageWords = 64 * kIdxLaneWords;  // per wavefront
// R1D: the 1D Lorenzo reconstruction done in the same pass (a segment holds
// whole blocks for every B), writing floats instead of codes.
template <bool T16, bool R1D>
__global__ void __launch_bounds__(256) k_decode_indexed(DecodeArgs a, const uint64_t* __restrict__ index,
                                                        IdxLayout L, uint64_t total_bits, uint16_t* __restrict__ codes,
                                                        float* __restrict__ sparse, Recon1D r, DecSummary* sum) {
    {  // workgroups k_decode_indexed_staged has decoded (the whole workgroup)
        StreamView sv0;
        sv0.setup(a.stream, a.stream_bits);
        if (idx_span(index, L, total_bits, sv0, blockIdx.x).fits) return;
    }
    // symbols per lane between flushes (16 words of stage either way) and
    // per 16-byte piece of output
    constexpr uint32_t kFlush = R1D ? 16 : kIdxFlush;
    constexpr uint32_t kPer16 = R1D ? 4 : 8;
    if (no_tables(a)) return;
    extern __shared__ __align__(16) uint32_t lds[];
    Decoder<T16> dec;
    TableCopy<T16, false, 256> tc;
    tc.fetch(a);
    const uint32_t tw = dec.attach(lds, a, tc.n_sub);
    tc.put(lds);
    const uint32_t lane = threadIdx.x & 63;
    uint32_t* stage = lds + tw + (threadIdx.x >> 6) * kIdxStageWords;
    lds_sync();
    const uint64_t g = blockIdx.x * 256ull + threadIdx.x;
    const uint64_t gw = g - lane;  // the wavefront's first segment
    const uint64_t nseg = L.nseg;
    const bool live = g < nseg;
    StreamView sv;
    sv.setup(a.stream, a.stream_bits);
    const uint64_t s0 = g * kIdxSeg;
    const uint32_t ns = live ? (uint32_t)min<uint64_t>(kIdxSeg, a.n - s0) : 0u;
    const uint64_t* grp = index + L.grp;
    const uint32_t* rel_bits = reinterpret_cast<const uint32_t*>(index + L.rel_bits);
    const uint16_t* rel_outs = reinterpret_cast<const uint16_t*>(index + L.rel_outs);
    auto first_bit = [&](uint64_t h) { return grp[2 * (h / kIdxGroup)] + rel_bits[h]; };
    const uint64_t start = live ? first_bit(g) : 0;
    const uint64_t end = !live ? 0 : g + 1 < nseg ? first_bit(g + 1) : total_bits;
    uint64_t rank = live ? grp[2 * (g / kIdxGroup) + 1] + rel_outs[g] : 0;
    bool bad = start > end || end > a.stream_bits;
    const uint64_t abit = start + sv.shift0;
    CursorWin cw;
    cw.sv = sv;
    cw.w0 = abit >> 5;
    cw.b0 = 0;
    cw.buf = live ? ((uint64_t)sv.word(cw.w0) << 32) | sv.word(cw.w0 + 1) : 0;
    // refill words come from 16-byte groups: the current one and the next,
    // already loaded (about 14 codewords of decode ahead of their use)
    auto load4 = [&](uint64_t q) -> uint4 {
        if (16 * (q + 1) <= sv.nbytes) {
            const U32x4 v = ((GlobalU32x4)sv.base)[q];
            return make_uint4(__builtin_bswap32(v.x), __builtin_bswap32(v.y), __builtin_bswap32(v.z),
                              __builtin_bswap32(v.w));
        }
        return make_uint4(sv.word(4 * q), sv.word(4 * q + 1), sv.word(4 * q + 2), sv.word(4 * q + 3));
    };
    uint64_t q4 = (cw.w0 + 2) >> 2;
    uint32_t qi = (uint32_t)((cw.w0 + 2) & 3);
    uint4 cur4 = make_uint4(0, 0, 0, 0), nxt4 = make_uint4(0, 0, 0, 0);
    if (live) {
        cur4 = load4(q4);
        nxt4 = load4(q4 + 1);
    }
    q4 += 2;
    uint32_t lp = (uint32_t)(abit & 31);
    float sprev = 0.f;  // R1D: the previous element's value in the block
    // the wavefront's segments lie kIdxSeg symbols apart; the last field
    // segment may be short, and only its whole pieces go through the stage
    for (uint32_t f0 = 0; f0 < kIdxSeg; f0 += kFlush) {
#pragma unroll
        for (uint32_t u = f0; u < f0 + kFlush; u += 8) {
            // Every lane decodes 8 codewords; a lane whose (last, short)
            // segment has ended keeps decoding at its end position (nothing
            // kept): its errors and outliers count only up to ns.  Outliers
            // wait for the end of the 8.
            uint32_t c[8];
            float o[8];
            uint32_t omask = 0;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                // one refill covers codewords of at most 32 bits (selects, no
                // branch); the 16-byte reload follows every fourth
                {
                    const bool need = lp - cw.b0 >= 32;
                    const uint32_t wv = qi == 0 ? cur4.x : qi == 1 ? cur4.y : qi == 2 ? cur4.z : cur4.w;
                    cw.buf = need ? (cw.buf << 32) | wv : cw.buf;
                    cw.b0 += need ? 32u : 0u;
                    qi += need ? 1u : 0u;
                    if (qi == 4) {
                        cur4 = nxt4;
                        nxt4 = load4(q4++);
                        qi = 0;
                    }
                }
                // after a longer codeword, more
                while (lp - cw.b0 >= 32) {
                    const uint32_t wv = qi == 0 ? cur4.x : qi == 1 ? cur4.y : qi == 2 ? cur4.z : cur4.w;
                    cw.buf = (cw.buf << 32) | wv;
                    cw.b0 += 32;
                    if (++qi == 4) {
                        cur4 = nxt4;
                        nxt4 = load4(q4++);
                        qi = 0;
                    }
                }
                // lp - cw.b0 < 32 here: the codeword's first 32 bits are in buf
                const uint32_t w = (uint32_t)((cw.buf << (lp - cw.b0)) >> 32);
                uint32_t len;
                const uint32_t sym = Decoder<T16>::sym(decode_one(dec, cw, w, lp, len));
                // past ns (or at an invalid codeword, an error) the lane
                // stays where it is: lp ends at the segment's end
                const bool in = u + k < ns;
                bad |= in & (len == 0);
                lp += in ? len : 0u;
                c[k] = sym;
                omask |= (uint32_t)(in & (sym == 0)) << k;
            }
            float ov[8];
#pragma unroll
            for (int k = 0; k < 8; k++) ov[k] = 0.f;
            if (omask) {
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    if ((omask >> k) & 1) {
                        float v = 0.f;
                        if (rank < a.n_outlier)
                            v = read_f32_bytes(a.outliers + 4 * rank);
                        else
                            bad = true;
                        rank++;
                        ov[k] = v;
                        if constexpr (!R1D) sparse[s0 + u + k] = v;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                o[k] = 0.f;
                if constexpr (R1D) {
                    // x_lorenzo_1d1l (src/dualquant.hh:915-931): a block's
                    // first element predicts from the halo (+0.0 or the
                    // block's pad value), the others from their predecessor
                    // (only for elements of the field: lanes past its end,
                    // whose values are dropped, must not index the halo,
                    // which has one entry per block of the field)
                    const uint64_t x = s0 + u + k;
                    if ((x % (uint64_t)r.B) == 0 && u + k < ns)
                        sprev = r.halo ? r.halo[r.halo_stride * (x / r.B) + 2] : 0.f;
                    const float sx = c[k] == 0 ? ov[k] : sprev + (float)((int32_t)c[k] - r.radius);
                    sprev = sx;
                    o[k] = (float)((double)sx * r.twoeb);
                }
            }
            uint32_t* d = stage + lane * kIdxLaneWords + (u - f0) * 16 / kFlush;
            if constexpr (R1D) {
#pragma unroll
                for (int k = 0; k < 8; k++) d[k] = __float_as_uint(o[k]);
            } else {
#pragma unroll
                for (int k = 0; k < 4; k++) d[k] = c[2 * k] | (c[2 * k + 1] << 16);
            }
            // pieces that end past a short last segment: straight out
            if (ns != kIdxSeg) {
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const uint32_t i = u + k;
                    if (i < ns && (i / kPer16 + 1) * kPer16 > ns) {
                        if constexpr (R1D)
                            r.out[s0 + i] = o[k];
                        else
                            codes[s0 + i] = (uint16_t)c[k];
                    }
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // piece i of this lane's store: lane q's piece j, slot lane + 64 i
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            const uint32_t slot = lane + 64 * i, q = slot / 4, j = slot % 4;
            const uint64_t gr = gw + q;
            const uint32_t nr = gr < nseg ? (uint32_t)min<uint64_t>(kIdxSeg, a.n - gr * kIdxSeg) : 0u;
            if (f0 + kPer16 * (j + 1) <= nr) {
                const uint32_t* w = stage + q * kIdxLaneWords + 4 * j;
                const uint4 val = make_uint4(w[0], w[1], w[2], w[3]);
                // codes and the 1D output are 16-byte aligned; gr * kIdxSeg + f0 + kPer16 * j is a
                // multiple of kPer16
                if constexpr (R1D)
                    *reinterpret_cast<uint4*>(r.out + gr * kIdxSeg + f0 + kPer16 * j) = val;
                else
                    *reinterpret_cast<uint4*>(codes + gr * kIdxSeg + f0 + kPer16 * j) = val;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // every segment ends where the next starts, the last at the stream's
    // last codeword bit
    if (live) bad |= 32 * cw.w0 + lp - sv.shift0 != end;
    if (bad) atomicOr(&sum->error, 1u);
}

// Decode with a decode index, the bits staged in LDS: the workgroup's 256
// segments are one contiguous span of the stream, staged with coalesced
// loads, and thread g decodes segment g out of LDS as the write pass decodes
// a subsequence.  A segment holds kIdxSeg = 128 symbols, 16 whole 16-byte
// units, so every thread writes its own units, in groups of four held in
// registers and stored back to back (R1D: the 1D reconstruction in the
// same pass, a segment holding whole blocks for every B, writing floats in
// groups of 16).  Workgroups whose span does not fit the stage return at
// once and leave their segments to k_decode_indexed.
template <bool T16, bool R1D>
__global__ void __launch_bounds__(256) k_decode_indexed_staged(DecodeArgs a, const uint64_t* __restrict__ index,
                                                               IdxLayout L, uint64_t total_bits,
                                                               uint16_t* __restrict__ codes,
                                                               float* __restrict__ sparse, Recon1D r,
                                                               DecSummary* sum) {
    StreamView sv;
    sv.setup(a.stream, a.stream_bits);
    const IdxSpan sp = idx_span(index, L, total_bits, sv, blockIdx.x);
    if (!sp.fits || no_tables(a)) return;  // (the whole workgroup)
    extern __shared__ __align__(16) uint32_t lds[];
    Decoder<T16> dec;
    uint32_t* stage;
    {
        TableCopy<T16, false, 256> tc;
        StageCopy<(kIdxSpanWords + 4 * 256 - 1) / (4 * 256), 256> sc;
        const uint32_t nvec = ((uint32_t)sp.nwords + 3) / 4;
        tc.fetch(a);
        sc.fetch(sv, sp.w_lo, nvec);
        stage = lds + dec.attach(lds, a, tc.n_sub);
        tc.put(lds);
        sc.put(stage, nvec);
    }
    lds_sync();
    const uint64_t g = blockIdx.x * 256ull + threadIdx.x;
    if (g >= L.nseg) return;  // no barrier follows
    const uint64_t* grp = index + L.grp;
    const uint32_t* rel_bits = reinterpret_cast<const uint32_t*>(index + L.rel_bits);
    const uint16_t* rel_outs = reinterpret_cast<const uint16_t*>(index + L.rel_outs);
    const uint64_t start = grp[2 * (g / kIdxGroup)] + rel_bits[g];
    const uint64_t end = g + 1 < L.nseg ? grp[2 * ((g + 1) / kIdxGroup)] + rel_bits[g + 1] : total_bits;
    uint64_t rank = grp[2 * (g / kIdxGroup) + 1] + rel_outs[g];
    const uint64_t s0 = g * kIdxSeg;
    const uint64_t span_lo = 32 * sp.w_lo;  // aligned-space bit of stage word 0
    // a segment outside the span (a damaged index) is an error, not decoded
    bool bad = start > end || end > a.stream_bits || start < sp.bs || end > sp.be;
    const uint32_t ns = bad ? 0u : (uint32_t)min<uint64_t>(kIdxSeg, a.n - s0);
    const RowWin win{stage};
    uint32_t lp = bad ? 0u : (uint32_t)(start + sv.shift0 - span_lo);
    // the loops count symbols, so an invalid codeword (len 0, an error)
    // needs no forced progress; a damaged stream stays within kIdxSpanOver
    // words past the span
    // one codeword, or two as the halves of a word
    auto next = [&]() -> uint32_t {
        uint32_t len;
        const uint32_t sym = Decoder<T16>::sym(decode_one(dec, win, win(lp), lp, len));
        if constexpr (!T16) bad |= len == 0;
        lp += len;
        return sym;
    };
    auto next2 = [&]() -> uint32_t {
        uint32_t e[2], l[2];
        decode_pair(dec, win, lp, e, l);
        if constexpr (!T16) bad |= (l[0] == 0) | (l[1] == 0);
        lp += l[0] + l[1];
        return Decoder<T16>::pack(e[0], e[1]);
    };
    auto outlier = [&](uint64_t i) {
        if (rank < a.n_outlier)
            sparse[i] = read_f32_bytes(a.outliers + 4 * rank);
        else
            bad = true;
        rank++;
    };
    if constexpr (R1D) {
        // x_lorenzo_1d1l (src/dualquant.hh:915-931), as in k_decode_indexed
        float sprev = 0.f;
        auto value = [&](uint32_t c, float ov, uint64_t x) -> float {
            if ((x % (uint64_t)r.B) == 0) sprev = r.halo ? r.halo[r.halo_stride * (x / r.B) + 2] : 0.f;
            const float sx = c == 0 ? ov : sprev + (float)((int32_t)c - r.radius);
            sprev = sx;
            return (float)((double)sx * r.twoeb);
        };
        const uint32_t nfull16 = ns & ~15u;
        for (uint32_t G = 0; G < nfull16; G += 16) {
            uint32_t c[16], least = ~0u;
#pragma unroll
            for (int k = 0; k < 16; k += 2) {
                const uint32_t w = next2();
                least = pk_min(least, w);
                c[k] = w & 0xFFFF;
                c[k + 1] = w >> 16;
            }
            float ov[16];
#pragma unroll
            for (int k = 0; k < 16; k++) ov[k] = 0.f;
            if (pk_has_zero(least)) {
#pragma unroll
                for (int k = 0; k < 16; k++) {
                    if (c[k] == 0) {
                        if (rank < a.n_outlier)
                            ov[k] = read_f32_bytes(a.outliers + 4 * rank);
                        else
                            bad = true;
                        rank++;
                    }
                }
            }
            float o[16];
#pragma unroll
            for (int k = 0; k < 16; k++) o[k] = value(c[k], ov[k], s0 + G + k);
#pragma unroll
            for (int q = 0; q < 4; q++)
                *reinterpret_cast<float4*>(r.out + s0 + G + 4 * q) =
                    make_float4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
        }
        for (uint32_t i = nfull16; i < ns; i++) {  // the field's last, partial group
            const uint32_t c = next();
            float ov = 0.f;
            if (c == 0) {
                if (rank < a.n_outlier)
                    ov = read_f32_bytes(a.outliers + 4 * rank);
                else
                    bad = true;
                rank++;
            }
            r.out[s0 + i] = value(c, ov, s0 + i);
        }
    } else {
        const uint32_t nfull = ns & ~7u;  // whole units
        for (uint32_t G = 0; G < nfull; G += 32) {
            // outliers are rare: one test per group, then in symbol order
            uint32_t w[16], least = ~0u;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const bool mine = G + 8 * u < nfull;  // differs across lanes only for the field's last segment
#pragma unroll
                for (int m = 0; m < 4; m++) w[4 * u + m] = ~0u;
                if (mine) {
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        w[4 * u + m] = next2();
                        least = pk_min(least, w[4 * u + m]);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (G + 8 * u < nfull)
                    *reinterpret_cast<uint4*>(codes + s0 + G + 8 * u) =
                        make_uint4(w[4 * u], w[4 * u + 1], w[4 * u + 2], w[4 * u + 3]);
            if (pk_has_zero(least)) {
#pragma unroll
                for (int k = 0; k < 32; k++)
                    if (((w[k / 2] >> (16 * (k & 1))) & 0xFFFF) == 0) outlier(s0 + G + k);
            }
        }
        for (uint32_t i = nfull; i < ns; i++) {  // the field's last, partial unit
            const uint32_t sym = next();
            codes[s0 + i] = (uint16_t)sym;
            if (sym == 0) outlier(s0 + i);
        }
    }
    // the segment ends where the next one starts
    if (!bad) bad = span_lo + lp - sv.shift0 != end;
    if (bad) atomicOr(&sum->error, 1u);
}

// Codewords and zeros of each write unit (kWriteWg consecutive subsequences),
// a wavefront per unit: sums[2 u], sums[2 u + 1].  A batch's units are
// numbered across its fields.
constexpr uint32_t kWriteWg = 512;
static_assert(kWriteWg % 64 == 0, "a unit is whole wavefronts");
__device__ __forceinline__ void decode_sums_unit(const uint32_t* __restrict__ cz, uint64_t nsub, uint64_t unit,
                                                 uint64_t* __restrict__ sums) {
    const uint32_t lane = lane_id2();
    uint32_t c = 0, z = 0;
#pragma unroll
    for (uint32_t i = 0; i < kWriteWg / 64; i++) {
        const uint64_t j = unit * kWriteWg + i * 64 + lane;
        const uint32_t v = j < nsub ? cz[j] : 0u;
        c += v & 0xFFFF;
        z += v >> 16;
    }
    c = wave_scan_dpp(c);
    z = wave_scan_dpp(z);
    if (lane == 63) {
        sums[0] = c;
        sums[1] = z;
    }
}
__global__ void __launch_bounds__(256) k_decode_sums(SubState s, uint64_t nsub, uint64_t nunits,
                                                     uint64_t* __restrict__ sums, const uint32_t* guard) {
    if (listed(guard)) return;
    const uint64_t u = blockIdx.x * 4ull + (threadIdx.x >> 6);
    if (u < nunits) decode_sums_unit(s.cz, nsub, u, sums + 2 * u);
}

// Exclusive prefixes of nunits pairs in place, the totals behind the last
// (one workgroup, kScanUnits pairs per thread and round).
constexpr uint32_t kScanUnits = 8;
__global__ void __launch_bounds__(1024) k_decode_scan(uint64_t* __restrict__ off, uint64_t nunits, const uint32_t* guard) {
    if (listed(guard)) return;
    __shared__ uint64_t sh[2][16];
    const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6;
    uint64_t carry[2] = {0, 0};
    for (uint64_t base = 0; base < nunits; base += 1024 * kScanUnits) {
        const uint64_t u0 = base + t * kScanUnits;
        uint64_t v[kScanUnits][2], run[2] = {0, 0};
#pragma unroll
        for (uint32_t i = 0; i < kScanUnits; i++)
            for (int q = 0; q < 2; q++) v[i][q] = u0 + i < nunits ? off[2 * (u0 + i) + q] : 0;
#pragma unroll
        for (uint32_t i = 0; i < kScanUnits; i++)
            for (int q = 0; q < 2; q++) {
                const uint64_t x = v[i][q];
                v[i][q] = run[q];  // before unit u0 + i, from u0
                run[q] += x;
            }
        uint64_t pre[2] = {run[0], run[1]};
#pragma unroll
        for (int d = 1; d < 64; d <<= 1)
            for (int q = 0; q < 2; q++) {
                const uint64_t x = __shfl_up(pre[q], d);
                if (lane >= (uint32_t)d) pre[q] += x;
            }
        if (lane == 63) {
            sh[0][w] = pre[0];
            sh[1][w] = pre[1];
        }
        lds_sync();
        uint64_t tot[2] = {0, 0};
        for (int q = 0; q < 2; q++) {
            pre[q] += carry[q] - run[q];
            for (uint32_t i = 0; i < 16; i++) {
                if (i < w) pre[q] += sh[q][i];
                tot[q] += sh[q][i];
            }
        }
        lds_sync();
#pragma unroll
        for (uint32_t i = 0; i < kScanUnits; i++)
            if (u0 + i < nunits)
                for (int q = 0; q < 2; q++) off[2 * (u0 + i) + q] = pre[q] + v[i][q];
        for (int q = 0; q < 2; q++) carry[q] += tot[q];
    }
    if (t < 2) off[2 * nunits + t] = carry[t];
}

// Both for a few units, in one launch of one workgroup (a launch and its gap
// are about 5 us, a wavefront's unit about 1: decode_scan stage 10.4 -> 6.0 us at
// 25 x 25 x 26).
constexpr uint64_t kOneOffsets = 64;
__global__ void __launch_bounds__(1024) k_decode_offsets(SubState s, uint64_t nsub, uint32_t nunits,
                                                         uint64_t* __restrict__ off, const uint32_t* guard) {
    if (listed(guard)) return;  // (the same for every wavefront)
    __shared__ uint64_t sums[2 * kOneOffsets];
    const uint32_t t = threadIdx.x;
    for (uint32_t u = t >> 6; u < nunits; u += 16) decode_sums_unit(s.cz, nsub, u, sums + 2 * u);
    lds_sync();
    if (t > nunits) return;
    uint64_t c = 0, z = 0;
    for (uint32_t i = 0; i < t; i++) c += sums[2 * i], z += sums[2 * i + 1];
    off[2 * t] = c;
    off[2 * t + 1] = z;
}

// Final decode.  Thread j decodes the codewords of subsequence j from its
// true start out of the workgroup's staged bits: its symbols are [O, E), O
// the unit's offset plus a scan of the unit's counts.
// Output goes out in whole 16-byte units of 8 symbols: the thread whose range
// holds a unit's first symbol writes the unit, decoding on past E into the
// following subsequences where the unit ends beyond it (the decode is on the
// true path there), and skips the symbols before its first unit (written by
// a predecessor).  Only the field's last unit may be partial.
constexpr uint32_t kWriteStageWords = kWriteWg * kSubWords + 32;  // + up to 7 codewords past the last range
constexpr uint32_t kWriteStageLds = kWriteStageWords + kWriteStageWords / kSubWords + 1;
constexpr uint32_t kWriteLdsWords = 1 + kWriteStageLds + 2 * (kWriteWg / 64);  // dynamic LDS after the tables
// base, off: the field's first unit's offsets and this unit's (field_base of
// a batch's earlier fields is subtracted).
template <bool T16>
__device__ __forceinline__ void decode_write_unit(const DecodeArgs& a, const SubState& s,
                                                  const uint64_t* __restrict__ base, const uint64_t* __restrict__ off,
                                                  uint16_t* __restrict__ codes, float* __restrict__ sparse,
                                                  DecSummary* sum, uint64_t unit) {
    extern __shared__ __align__(16) uint32_t lds[];
    Decoder<T16> dec;
    uint32_t* st;
    StreamView sv;
    sv.setup(a.stream, a.stream_bits);
    const uint64_t J0 = unit * kWriteWg;
    const uint64_t j = J0 + threadIdx.x;
    const bool live = j < a.nsub;
    uint32_t cz, first;
    {
        TableCopy<T16, false, kWriteWg> tc;
        StageCopy<(kWriteStageWords + 4 * kWriteWg - 1) / (4 * kWriteWg), kWriteWg> sc;
        tc.fetch(a);
        sc.fetch(sv, J0 * kSubWords, (kWriteStageWords + 3) / 4);
        cz = live ? s.cz[j] : 0u;
        first = live ? s.b[j] : 0u;
        st = lds + dec.attach(lds, a, tc.n_sub) + 1;
        tc.put(lds);
        sc.put_rows(st, kWriteStageWords);
    }
    uint32_t* wsum = st + kWriteStageLds;  // counts and zeros of each wavefront
    const uint32_t ic = wave_scan_dpp(cz & 0xFFFF), iz = wave_scan_dpp(cz >> 16);
    const uint32_t w = threadIdx.x >> 6;
    if (lane_id2() == 63) {
        wsum[2 * w] = ic;
        wsum[2 * w + 1] = iz;
    }
    lds_sync();
    if (!live) return;
    uint64_t O = off[0] - base[0] + ic - (cz & 0xFFFF);
    uint64_t rank = off[1] - base[1] + iz - (cz >> 16);
    for (uint32_t i = 0; i < w; i++) {
        O += wsum[2 * i];
        rank += wsum[2 * i + 1];
    }
    const uint64_t E = min<uint64_t>(O + (cz & 0xFFFF), a.n);
    uint32_t lp = threadIdx.x * kSubBits + first + sv.shift0;
    bool bad = false;
    // the loops below count symbols, so an invalid codeword (len 0, an
    // error) needs no forced progress
    const PadWin win{st};
    // one codeword, or two as the halves of a word
    auto next = [&]() -> uint32_t {
        uint32_t len;
        const uint32_t sym = Decoder<T16>::sym(decode_one(dec, win, win(lp), lp, len));
        if constexpr (!T16) bad |= len == 0;
        lp += len;
        return sym;
    };
    auto next2 = [&]() -> uint32_t {
        uint32_t e[2], l[2];
        decode_pair(dec, win, lp, e, l);
        if constexpr (!T16) bad |= (l[0] == 0) | (l[1] == 0);
        lp += l[0] + l[1];
        return Decoder<T16>::pack(e[0], e[1]);
    };
    auto outlier = [&](uint64_t i) {
        if (rank < a.n_outlier)
            sparse[i] = read_f32_bytes(a.outliers + 4 * rank);
        else
            bad = true;
        rank++;
    };
    const uint64_t W0 = (O + 7) & ~7ull;  // this thread's first unit
    uint64_t i = O;
    for (; i < E && i < W0; i++)          // a predecessor's unit: decode, count zeros, skip
        rank += next() == 0;
    if (W0 < E) {
        const uint64_t W1 = min<uint64_t>((E + 7) & ~7ull, a.n);
        const uint64_t Wf = W0 + ((W1 - W0) & ~7ull);  // end of the whole units
        // Whole units go out in groups of four (64 bytes) held in registers
        // and stored back to back: the L2 then sees long runs of each lane's
        // output, where units stored as they were decoded left partially
        // written lines that were written back several times.  Groups start
        // at the lane's first unit, so only its last group is partial.
        for (uint64_t G = W0; G < Wf; G += 32) {
            // outliers are rare: one test per group, then in symbol order
            uint32_t w[16], least = ~0u;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint64_t iu = G + 8 * u;
                const bool mine = iu < Wf;  // differs across lanes only in a last group
#pragma unroll
                for (int m = 0; m < 4; m++) w[4 * u + m] = ~0u;
                if (mine) {
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        w[4 * u + m] = next2();
                        least = pk_min(least, w[4 * u + m]);
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint64_t iu = G + 8 * u;
                if (iu < Wf)
                    *reinterpret_cast<uint4*>(codes + iu) =
                        make_uint4(w[4 * u], w[4 * u + 1], w[4 * u + 2], w[4 * u + 3]);
            }
            if (pk_has_zero(least)) {
#pragma unroll
                for (int k = 0; k < 32; k++)
                    if (((w[k / 2] >> (16 * (k & 1))) & 0xFFFF) == 0) outlier(G + k);
            }
        }
        i = Wf;
        for (; i < W1; i++) {  // the field's last, partial unit
            const uint32_t sym = next();
            codes[i] = (uint16_t)sym;
            if (sym == 0) outlier(i);
        }
    }
    if (bad) atomicOr(&sum->error, 1u);
}

template <bool T16>
__global__ void __launch_bounds__(kWriteWg) k_decode_write(DecodeArgs a, SubState s, const uint64_t* __restrict__ off,
                                                           uint16_t* __restrict__ codes, float* __restrict__ sparse,
                                                           DecSummary* sum, const uint32_t* guard) {
    if (listed(guard)) return;
    decode_write_unit<T16>(a, s, off, off + 2 * (uint64_t)blockIdx.x, codes, sparse, sum, blockIdx.x);
}

__global__ void k_fill_u16(uint16_t* p, uint64_t n, uint16_t v) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void k_scatter_all(const uint8_t* __restrict__ outl, uint64_t n, float* __restrict__ sparse) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        sparse[i] = read_f32_bytes(outl + 4 * i);
}

// ------------------------------------------------------------------ reconstruction

constexpr int32_t kExact = 1 << 21;

__device__ __forceinline__ float scale_out(int32_t s, double twoeb) { return (float)((double)(float)s * twoeb); }

// An outlier's s is its stored value itself, sign of zero included (a
// non-outlier s is never -0.0: pred + (float)(code - R) with a +0.0 addend).
__device__ __forceinline__ float scale_outlier(float v, double twoeb) { return (float)((double)v * twoeb); }

// Value of the lane D below, in the same row of 16 lanes (else 0): a DPP move,
// where __shfl_up is an LDS permute with an LDS round trip's latency on the
// scan's chain.
template <int D>
__device__ __forceinline__ int32_t lane_below(int32_t v) {
    return (int32_t)dpp_move<0x110 + D>((uint32_t)v);
}

// Inclusive segmented scan over segments of L lanes: v, and whether the lane
// or one before it in its segment starts a new run (f set).  Rows of 16 lanes
// first, then a segment's rows: row 0's last lane to row 1 and row 2's to row
// 3, and the last lane of the first two to the others.
template <int L, int D = 1>
__device__ __forceinline__ void seg_scan_lanes(int32_t& v, int32_t& f) {
    if constexpr (D < L) {
        int32_t nv, nf;  // (every lane is active here: 0 where it has no source)
        if constexpr (D < 16) {
            nv = lane_below<D>(v), nf = lane_below<D>(f);
            if (lane_id2() % L % 16 < (uint32_t)D) nv = nf = 0;
        } else if constexpr (D == 16) {
            nv = (int32_t)dpp_move<0x142, 0xA>((uint32_t)v), nf = (int32_t)dpp_move<0x142, 0xA>((uint32_t)f);
        } else {
            nv = (int32_t)dpp_move<0x143, 0xC>((uint32_t)v), nf = (int32_t)dpp_move<0x143, 0xC>((uint32_t)f);
        }
        if (!f) v += nv;
        f |= nf;
        seg_scan_lanes<L, 2 * D>(v, f);
    }
}
template <int B>
__device__ __forceinline__ int32_t seg_scan(int32_t v, bool f) {
    int32_t g = f;
    seg_scan_lanes<B>(v, g);
    return v;
}

__device__ __forceinline__ bool exact_outlier(float v) { return v == __builtin_rintf(v) && __builtin_fabsf(v) < (float)kExact; }

__device__ __forceinline__ void flag_blocks(bool bad, int B, uint64_t blk_x0, uint64_t by, uint64_t bz, uint64_t nbx,
                                            uint64_t nby, uint32_t* flagged, uint32_t* nflagged) {
    const uint64_t m = __ballot(bad);
    if (!m) return;
    const uint32_t lane = lane_id2();
    if (lane % B == 0) {
        const uint64_t seg = (B == 64) ? ~0ull : (((1ull << B) - 1) << lane);
        if (m & seg) {
            const uint64_t bx = blk_x0 + lane / B;
            const uint64_t id = bx + nbx * (by + nby * bz);
            const uint32_t slot = atomicAdd(nflagged, 1u);
            flagged[slot] = (uint32_t)id;
        }
    }
}

// Halo values of the block holding x, for the integer recurrences: exact
// when every one is an integer below kExact (else the block is listed).
struct IHalo {
    int32_t z, y, x;
    bool exact;
};
__device__ __forceinline__ IHalo load_ihalo(const ReconArgs& a, bool xin, uint64_t x, int B, uint64_t by,
                                            uint64_t bz) {
    IHalo h{0, 0, 0, true};
    if (xin) {
        const float* p = a.halo + a.halo_stride * ((x / B) + a.hb0 * (by + a.hb1 * bz));
        h.exact = exact_outlier(p[0]) && exact_outlier(p[1]) && exact_outlier(p[2]);
        h.z = h.exact ? (int32_t)p[0] : 0;
        h.y = h.exact ? (int32_t)p[1] : 0;
        h.x = h.exact ? (int32_t)p[2] : 0;
    }
    return h;
}

// PAD: with halo values h (x_block_pad / x_edge_pad), r = s - Y - Z + YZ
// is still a running sum along x, with Y, Z, YZ read from the halo faces in
// the first row / plane of the block and a start of h.x - h.y in the block's
// first row of its first plane (the only row where X - XY - XZ + XYZ of the
// halo does not cancel).
template <int B, bool PAD>
__device__ __forceinline__ void recon_3d_tile(uint64_t t, const uint16_t* __restrict__ codes, const float* __restrict__ sparse,
                                                  float* __restrict__ out, const ReconArgs& a, uint32_t* flagged,
                                                  uint32_t* nflagged) {
    const uint32_t lane = lane_id2();
    const uint64_t sy = a.d0, sz = a.d0 * a.d1;
    const uint64_t nbx = (a.d0 + B - 1) / B, nby = (a.d1 + B - 1) / B;
    {
        const uint64_t tx = t % a.ntiles_x;
        const uint64_t ty = (t / a.ntiles_x) % a.ntiles_y;
        const uint64_t tz = t / (a.ntiles_x * a.ntiles_y);
        const uint64_t x = tx * 64 + lane;
        const uint64_t y0 = ty * B, z0 = tz * B;
        const bool xin = x < a.d0;
        const bool bstart = (lane % B) == 0;
        bool bad = false;
        IHalo h{0, 0, 0, true};
        if constexpr (PAD) {
            h = load_ihalo(a, xin, x, B, ty, tz);
            bad = !h.exact;
        }
        int32_t prevplane[B];
#pragma unroll
        for (int j = 0; j < B; j++) prevplane[j] = 0;
        auto load = [&](int zz, int yy) -> uint32_t {
            return xin && zz < B && z0 + zz < a.d2 && y0 + yy < a.d1 ? codes[x + (y0 + yy) * sy + (z0 + zz) * sz]
                                                                     : (uint32_t)a.radius;
        };
        RowsAhead<uint32_t> rows;
        rows.ahead([&](int r) { return load(0, r); });
        for (int zz = 0; zz < B; zz++) {
            const uint64_t z = z0 + zz;
            if (z >= a.d2) break;
            int32_t srow = 0, zrow = 0;
#pragma unroll
            for (int yy = 0; yy < B; yy++) {
                const uint64_t y = y0 + yy;
                if (yy % kRowsAhead == 0) {
                    rows.take();
                    const int ny = yy + kRowsAhead < B ? yy + kRowsAhead : 0;
                    rows.ahead([&](int r) { return load(ny ? zz : zz + 1, ny + r); });
                }
                if (y < a.d1) {
                    const uint64_t idx = x + y * sy + z * sz;
                    const uint32_t c = rows.cur[yy % kRowsAhead];
                    const bool isout = xin && c == 0;
                    const int32_t Y = yy > 0 ? srow : h.y;
                    const int32_t Z = zz > 0 ? prevplane[yy] : h.z;
                    const int32_t YZ = (yy > 0 && zz > 0) ? zrow : (zz == 0 ? h.z : h.y);
                    int32_t g0;
                    float v = 0.f;
                    if (isout) {
                        v = sparse[idx];
                        if (!exact_outlier(v)) bad = true;
                        g0 = (int32_t)v - Y - Z + YZ;
                    } else {
                        g0 = (int32_t)c - a.radius;
                        if (PAD && bstart && zz == 0 && yy == 0) g0 += h.x - h.y;
                    }
                    const int32_t G = seg_scan<B>(g0, isout || bstart);
                    const int32_t sv = G + Y + Z - YZ;
                    if (sv >= kExact || sv <= -kExact) bad = true;
                    if (xin) out[idx] = isout ? scale_outlier(v, a.twoeb) : scale_out(sv, a.twoeb);
                    zrow = Z;
                    prevplane[yy] = sv;
                    srow = sv;
                }
            }
        }
        flag_blocks(bad, B, tx * (64 / B), ty, tz, nbx, nby, flagged, nflagged);
    }
}

template <int B, bool PAD = false>
__global__ void __launch_bounds__(256) k_recon_3d(const uint16_t* __restrict__ codes, const float* __restrict__ sparse,
                                                  float* __restrict__ out, ReconArgs a, uint32_t* flagged,
                                                  uint32_t* nflagged) {
    if (listed(a.guard)) return;  // decode output not final: a later launch redoes this
    const uint64_t ntiles = a.ntiles_x * a.ntiles_y * a.ntiles_z;
    const uint64_t wave = blockIdx.x * 4ull + (threadIdx.x >> 6);
    const uint64_t nwaves = gridDim.x * 4ull;
    for (uint64_t t = wave; t < ntiles; t += nwaves) recon_3d_tile<B, PAD>(t, codes, sparse, out, a, flagged, nflagged);
}

// PAD: r = s - N runs along x from 0 at the block start (W - NW of the
// x-face halo cancels), with N = h.y in the block's first row.
template <int B, bool PAD>
__device__ __forceinline__ void recon_2d_tile(uint64_t t, const uint16_t* __restrict__ codes, const float* __restrict__ sparse,
                                                  float* __restrict__ out, const ReconArgs& a, uint32_t* flagged,
                                                  uint32_t* nflagged) {
    const uint32_t lane = lane_id2();
    const uint64_t nbx = (a.d0 + B - 1) / B, nby = (a.d1 + B - 1) / B;
    {
        const uint64_t tx = t % a.ntiles_x;
        const uint64_t ty = t / a.ntiles_x;
        const uint64_t x = tx * 64 + lane;
        const uint64_t y0 = ty * B;
        const bool xin = x < a.d0;
        const bool bstart = (lane % B) == 0;
        bool bad = false;
        IHalo h{0, 0, 0, true};
        if constexpr (PAD) {
            h = load_ihalo(a, xin, x, B, ty, 0);
            bad = !h.exact;
        }
        int32_t srow = 0;
        auto load = [&](int yy) -> uint32_t {
            return xin && yy < B && y0 + yy < a.d1 ? codes[x + (y0 + yy) * a.d0] : (uint32_t)a.radius;
        };
        RowsAhead<uint32_t> rows;
        rows.ahead([&](int r) { return load(r); });
#pragma unroll
        for (int yy = 0; yy < B; yy++) {
            const uint64_t y = y0 + yy;
            if (yy % kRowsAhead == 0) {
                rows.take();
                rows.ahead([&](int r) { return load(yy + kRowsAhead + r); });
            }
            if (y < a.d1) {
                const uint64_t idx = x + y * a.d0;
                const uint32_t c = rows.cur[yy % kRowsAhead];
                const bool isout = xin && c == 0;
                const int32_t N = yy > 0 ? srow : h.y;
                int32_t g0;
                float v = 0.f;
                if (isout) {
                    v = sparse[idx];
                    if (!exact_outlier(v)) bad = true;
                    g0 = (int32_t)v - N;
                } else {
                    g0 = (int32_t)c - a.radius;
                }
                const int32_t G = seg_scan<B>(g0, isout || bstart);
                const int32_t sv = G + N;
                if (sv >= kExact || sv <= -kExact) bad = true;
                if (xin) out[idx] = isout ? scale_outlier(v, a.twoeb) : scale_out(sv, a.twoeb);
                srow = sv;
            }
        }
        flag_blocks(bad, B, tx * (64 / B), ty, 0, nbx, nby, flagged, nflagged);
    }
}

template <int B, bool PAD = false>
__global__ void __launch_bounds__(256) k_recon_2d(const uint16_t* __restrict__ codes, const float* __restrict__ sparse,
                                                  float* __restrict__ out, ReconArgs a, uint32_t* flagged,
                                                  uint32_t* nflagged) {
    if (listed(a.guard)) return;  // decode output not final: a later launch redoes this
    const uint64_t ntiles = a.ntiles_x * a.ntiles_y;
    const uint64_t wave = blockIdx.x * 4ull + (threadIdx.x >> 6);
    const uint64_t nwaves = gridDim.x * 4ull;
    for (uint64_t t = wave; t < ntiles; t += nwaves) recon_2d_tile<B, PAD>(t, codes, sparse, out, a, flagged, nflagged);
}

// PAD: the running sum starts from the block's pad value (a raw, usually
// non-integral value for 1D block / edge padding: such blocks are listed).
template <int B, bool PAD>
__device__ __forceinline__ void recon_1d_tile(uint64_t t, const uint16_t* __restrict__ codes, const float* __restrict__ sparse,
                                                  float* __restrict__ out, const ReconArgs& a, uint32_t* flagged,
                                                  uint32_t* nflagged) {
    const uint32_t lane = lane_id2();
    const uint64_t nbx = (a.d0 + B - 1) / B;
    {
        const uint64_t x = t * 64 + lane;
        const bool xin = x < a.d0;
        const bool bstart = (lane % B) == 0;
        bool bad = false;
        IHalo h{0, 0, 0, true};
        if constexpr (PAD) {
            h = load_ihalo(a, xin, x, B, 0, 0);
            bad = !h.exact;
        }
        const uint32_t c = xin ? codes[x] : (uint32_t)a.radius;
        const bool isout = xin && c == 0;
        int32_t g0;
        float v = 0.f;
        if (isout) {
            v = sparse[x];
            if (!exact_outlier(v)) bad = true;
            g0 = (int32_t)v;
        } else {
            g0 = (int32_t)c - a.radius;
            if (PAD && bstart) g0 += h.x;
        }
        const int32_t sv = seg_scan<B>(g0, isout || bstart);
        if (sv >= kExact || sv <= -kExact) bad = true;
        if (xin) out[x] = isout ? scale_outlier(v, a.twoeb) : scale_out(sv, a.twoeb);
        flag_blocks(bad, B, t * (64 / B), 0, 0, nbx, 1, flagged, nflagged);
    }
}

template <int B, bool PAD = false>
__global__ void __launch_bounds__(256) k_recon_1d(const uint16_t* __restrict__ codes, const float* __restrict__ sparse,
                                                  float* __restrict__ out, ReconArgs a, uint32_t* flagged,
                                                  uint32_t* nflagged) {
    if (listed(a.guard)) return;  // decode output not final: a later launch redoes this
    const uint64_t ntiles = a.ntiles_x;
    const uint64_t wave = blockIdx.x * 4ull + (threadIdx.x >> 6);
    const uint64_t nwaves = gridDim.x * 4ull;
    for (uint64_t t = wave; t < ntiles; t += nwaves) recon_1d_tile<B, PAD>(t, codes, sparse, out, a, flagged, nflagged);
}

// One thread per listed block: the reference's sequential fp32 recurrence in
// its own association, using the block's region of `out` for the s values
// before scaling them in place.
// Listed blocks i0, i0 + di, ... of one field.
__device__ __forceinline__ void recon_fallback_blocks(int ndim, int B, const uint16_t* __restrict__ codes,
                                                      const float* __restrict__ sparse, float* __restrict__ out,
                                                      const ReconArgs& a, const uint32_t* __restrict__ flagged,
                                                      const uint32_t* __restrict__ nflagged, uint64_t i0, uint64_t di) {
    const uint32_t nl = *nflagged;
    const uint64_t nbx = (a.d0 + B - 1) / B, nby = (a.d1 + B - 1) / B;
    const uint64_t sy = a.d0, sz = a.d0 * a.d1;
    for (uint64_t i = i0; i < nl; i += di) {
        const uint64_t id = flagged[i];
        const uint64_t bx = id % nbx, by = (id / nbx) % nby, bz = id / (nbx * nby);
        const uint64_t x0 = bx * B, y0 = by * B, z0 = bz * B;
        // halo cells: z face, else y face, else x face in 3D; x face, else y in 2D
        float hz = 0.f, hy = 0.f, hx = 0.f;
        if (a.halo) {
            const float* hp = a.halo + a.halo_stride * (bx + a.hb0 * (by + a.hb1 * bz));
            hz = hp[0];
            hy = hp[1];
            hx = hp[2];
        }
        const uint64_t xe = min(x0 + B, a.d0), ye = min(y0 + B, a.d1), ze = min(z0 + B, a.d2);
        for (uint64_t z = z0; z < ze; z++)
            for (uint64_t y = y0; y < ye; y++)
                for (uint64_t x = x0; x < xe; x++) {
                    const uint64_t idx = x + y * sy + z * sz;
                    const bool ix = x > x0, iy = y > y0, iz = z > z0;  // neighbour inside the block
                    float pred;
                    if (ndim == 1) {
                        pred = ix ? out[idx - 1] : hx;
                    } else if (ndim == 2) {
                        const float W = ix ? out[idx - 1] : hx;
                        const float N = iy ? out[idx - sy] : hy;
                        const float NW = (ix && iy) ? out[idx - 1 - sy] : (!ix ? hx : hy);
                        pred = N + W;
                        pred = pred - NW;
                    } else {
                        const float X = ix ? out[idx - 1] : hx;
                        const float Y = iy ? out[idx - sy] : hy;
                        const float Z = iz ? out[idx - sz] : hz;
                        const float XY = (ix && iy) ? out[idx - 1 - sy] : (!iy ? hy : hx);
                        const float XZ = (ix && iz) ? out[idx - 1 - sz] : (!iz ? hz : hx);
                        const float YZ = (iy && iz) ? out[idx - sy - sz] : (!iz ? hz : hy);
                        const float XYZ = (ix && iy && iz) ? out[idx - 1 - sy - sz] : (!iz ? hz : !iy ? hy : hx);
                        pred = XYZ - XY;
                        pred = pred - XZ;
                        pred = pred - YZ;
                        pred = pred + X;
                        pred = pred + Y;
                        pred = pred + Z;
                    }
                    const uint32_t c = codes[idx];
                    out[idx] = c == 0 ? sparse[idx] : pred + (float)((int32_t)c - a.radius);
                }
        for (uint64_t z = z0; z < ze; z++)
            for (uint64_t y = y0; y < ye; y++)
                for (uint64_t x = x0; x < xe; x++) {
                    const uint64_t idx = x + y * sy + z * sz;
                    out[idx] = (float)((double)out[idx] * a.twoeb);
                }
    }
}

__global__ void __launch_bounds__(64) k_recon_fallback(int ndim, int B, const uint16_t* __restrict__ codes,
                                                       const float* __restrict__ sparse, float* __restrict__ out,
                                                       ReconArgs a, const uint32_t* __restrict__ flagged,
                                                       const uint32_t* __restrict__ nflagged) {
    if (listed(a.guard)) return;  // decode output not final: a later launch redoes this
    recon_fallback_blocks(ndim, B, codes, sparse, out, a, flagged, nflagged,
                          blockIdx.x * (uint64_t)blockDim.x + threadIdx.x, (uint64_t)gridDim.x * blockDim.x);
}

// Four consecutive x per lane (8-byte code loads, 16-byte stores).  A block
// row of B elements spans B/4 lanes: each lane runs the Lorenzo prefix over
// its four elements sequentially, then a segmented scan over the lanes of the
// row carries the running value in, up to the lane's first restart (an
// outlier or the block start).
template <int B>
__device__ __forceinline__ void row_scan4(int32_t (&D)[4], const int32_t (&g)[4], const bool (&rs)[4]) {
    constexpr int L = B / 4;
    D[0] = g[0];
#pragma unroll
    for (int i = 1; i < 4; i++) D[i] = rs[i] ? g[i] : D[i - 1] + g[i];
    if constexpr (L > 1) {
        int32_t T = D[3];
        int32_t f = rs[0] | rs[1] | rs[2] | rs[3];
        seg_scan_lanes<L>(T, f);
        int32_t carry = lane_below<1>(T);
        if (lane_id2() % L == 0) carry = 0;
        bool open = true;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            open = open && !rs[i];
            if (open) D[i] += carry;
        }
    }
}

// ALN: the x extent is a multiple of 4 and codes / output are 8- / 16-byte
// aligned, so a lane's four codes and outputs move as one uint2 / float4;
// otherwise element by element, elements past the row's end reading as the
// radius code (no change) and storing nothing.
template <int ND, int B, bool ALN>
__device__ __forceinline__ void recon_x4_tile(uint64_t t, const uint16_t* __restrict__ codes, const float* __restrict__ sparse,
                                                  float* __restrict__ out, const ReconArgs& a, uint32_t* flagged,
                                                  uint32_t* nflagged) {
    constexpr int L = B / 4;
    constexpr int YB = ND >= 2 ? B : 1;
    constexpr int ZB = ND >= 3 ? B : 1;
    const uint32_t lane = lane_id2();
    const uint64_t ntx = (a.d0 + 255) / 256;
    const uint64_t nty = ND >= 2 ? a.ntiles_y : 1;
    const uint64_t sy = a.d0, sz = a.d0 * a.d1;
    const uint64_t nbx = (a.d0 + B - 1) / B, nby = ND >= 2 ? (a.d1 + B - 1) / B : 1;
    const uint32_t R = (uint32_t)a.radius;
    {
        const uint64_t tx = t % ntx;
        const uint64_t ty = (t / ntx) % nty;
        const uint64_t tz = t / (ntx * nty);
        const uint64_t x0 = tx * 256 + 4 * lane;
        const bool xin = x0 < a.d0;  // ALN: all four or none
        bool ein[4];                 // element x0 + i inside the row
#pragma unroll
        for (int i = 0; i < 4; i++) ein[i] = ALN ? xin : x0 + i < a.d0;
        const bool rowstart = (lane % L) == 0;
        bool bad = false;
        int32_t prev[ZB > 1 ? B : 1][4];
#pragma unroll
        for (int j = 0; j < (ZB > 1 ? B : 1); j++)
#pragma unroll
            for (int i = 0; i < 4; i++) prev[j][i] = 0;
        // a row's four codes, two to a word (the radius code outside the field)
        auto load = [&](int zz, int yy) -> uint2 {
            const uint64_t y = ND >= 2 ? ty * B + yy : 0, z = ND >= 3 ? tz * B + zz : 0;
            uint2 cw = make_uint2(R | (R << 16), R | (R << 16));
            if (zz < ZB && yy < YB && y < a.d1 && z < a.d2) {
                const uint16_t* p = codes + x0 + y * sy + z * sz;
                if constexpr (ALN) {
                    if (xin) cw = *reinterpret_cast<const uint2*>(p);
                } else {
                    if (ein[3]) {
                        __builtin_memcpy(&cw, p, 8);
                    } else if (xin) {
                        cw.x = p[0] | ((ein[1] ? (uint32_t)p[1] : R) << 16);
                        if (ein[2]) cw.y = p[2] | (R << 16);
                    }
                }
            }
            return cw;
        };
        RowsAhead<uint2> rows;
        if constexpr (ND > 1) rows.ahead([&](int r) { return load(0, r); });
        for (int zz = 0; zz < ZB; zz++) {
            const uint64_t z = ND >= 3 ? tz * B + zz : 0;
            if (z >= a.d2) break;
            int32_t srow[4] = {0, 0, 0, 0}, zrow[4] = {0, 0, 0, 0};
#pragma unroll
            for (int yy = 0; yy < YB; yy++) {
                const uint64_t y = ND >= 2 ? ty * B + yy : 0;
                if (ND > 1 && yy % kRowsAhead == 0) {
                    rows.take();
                    const int ny = yy + kRowsAhead < YB ? yy + kRowsAhead : 0;
                    rows.ahead([&](int r) { return load(ny ? zz : zz + 1, ny + r); });
                }
                if (y < a.d1) {
                    const uint64_t idx = x0 + y * sy + z * sz;
                    const uint2 cw = ND > 1 ? rows.cur[yy % kRowsAhead] : load(0, 0);
                    const uint32_t c[4] = {cw.x & 0xFFFF, cw.x >> 16, cw.y & 0xFFFF, cw.y >> 16};
                    int32_t g[4], base[4], Zv[4], D[4];
                    bool rs[4], isout[4];
                    float v[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int32_t Y = (ND >= 2 && yy > 0) ? srow[i] : 0;
                        Zv[i] = (ND >= 3 && zz > 0) ? prev[ZB > 1 ? yy : 0][i] : 0;
                        const int32_t YZ = (ND >= 3 && yy > 0 && zz > 0) ? zrow[i] : 0;
                        base[i] = Y + Zv[i] - YZ;
                        isout[i] = ein[i] && c[i] == 0;
                        v[i] = 0.f;
                        g[i] = (int32_t)c[i] - a.radius;
                    }
                    // outliers are rare: one test for the lane's four elements
                    const bool anyout = isout[0] | isout[1] | isout[2] | isout[3];
                    if (anyout) {
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            if (isout[i]) {
                                v[i] = sparse[idx + i];
                                if (!exact_outlier(v[i])) bad = true;
                                g[i] = (int32_t)v[i] - base[i];
                            }
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) rs[i] = isout[i] || (i == 0 && rowstart);
                    row_scan4<B>(D, g, rs);
                    float o[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int32_t sv = D[i] + base[i];
                        if (sv >= kExact || sv <= -kExact) bad = true;
                        o[i] = scale_out(sv, a.twoeb);
                        if (ND >= 3) {
                            zrow[i] = Zv[i];
                            prev[ZB > 1 ? yy : 0][i] = sv;
                        }
                        srow[i] = sv;
                    }
                    if (anyout) {
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (isout[i]) o[i] = scale_outlier(v[i], a.twoeb);
                    }
                    if constexpr (ALN) {
                        if (xin) *reinterpret_cast<float4*>(out + idx) = make_float4(o[0], o[1], o[2], o[3]);
                    } else {
                        if (ein[3]) {
                            __builtin_memcpy(out + idx, o, 16);
                        } else {
#pragma unroll
                            for (int i = 0; i < 3; i++)
                                if (ein[i]) out[idx + i] = o[i];
                        }
                    }
                }
            }
        }
        flag_blocks(bad, L, tx * (256 / B), ty, tz, nbx, nby, flagged, nflagged);
    }
}

// (3D, B 8: four wavefronts per SIMD for a few spilled registers; with the
// 135 it would take, three, the 1 GiB field ran 371 -> 400 us.)
template <int ND, int B, bool ALN>
__global__ void __launch_bounds__(256, ND == 3 && B == 8 ? 4 : 1) k_recon_x4(const uint16_t* __restrict__ codes, const float* __restrict__ sparse,
                                                  float* __restrict__ out, ReconArgs a, uint32_t* flagged,
                                                  uint32_t* nflagged) {
    if (listed(a.guard)) return;  // decode output not final: a later launch redoes this
    const uint64_t ntx = (a.d0 + 255) / 256;
    const uint64_t nty = ND >= 2 ? a.ntiles_y : 1, ntz = ND >= 3 ? a.ntiles_z : 1;
    const uint64_t ntiles = ntx * nty * ntz;
    const uint64_t wave = blockIdx.x * 4ull + (threadIdx.x >> 6);
    const uint64_t nwaves = gridDim.x * 4ull;
    for (uint64_t t = wave; t < ntiles; t += nwaves)
        recon_x4_tile<ND, B, ALN>(t, codes, sparse, out, a, flagged, nflagged);
}

// ------------------------------------------------------------------ batched fields
//
// A batch decompress runs every stage once for all of its fields: each
// launch walks a queue of units that spans the fields (unit u belongs to
// field f when start[f] <= u < start[f + 1]) and runs the single-field body
// on the field's descriptor.  A unit is uniform across its workgroup (sync,
// write) or its wavefront (reconstruction), so the field lookup and the
// descriptor reads are scalar.

__global__ void __launch_bounds__(kSyncWg) k_decode_sync_multi(const DecField* __restrict__ fd,
                                                               const uint64_t* __restrict__ start, int nf) {
    const uint64_t u = blockIdx.x;
    const int f = field_of(start, nf, u);
    const DecodeArgs a = fd[f].a;
    const SubState s = fd[f].s;
    decode_sync_unit<true>(a, s, fd[f].sum, u - start[f], (uint32_t)u);
}

// Re-decode pass: a workgroup per sync unit, whose listed subsequences are one
// field's, so that the tables are in LDS.
__global__ void __launch_bounds__(256) k_decode_pass_multi(const DecField* __restrict__ fd,
                                                           const uint64_t* __restrict__ start, int nf, uint32_t pass) {
    const uint64_t u = blockIdx.x;
    const int f = field_of(start, nf, u);
    const DecodeArgs a = fd[f].a;
    const SubState s = fd[f].s;
    decode_pass_stripe<true>(a, s, pass, fd[f].sum, (uint32_t)u, 0, 1);
}

__global__ void __launch_bounds__(256) k_decode_sums_multi(const DecField* __restrict__ fd,
                                                           const uint64_t* __restrict__ start, int nf,
                                                           uint64_t* __restrict__ sums) {
    const uint64_t u = blockIdx.x * 4ull + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (u >= start[nf]) return;
    const int f = field_of(start, nf, u);
    decode_sums_unit(fd[f].s.cz, fd[f].a.nsub, u - start[f], sums + 2 * u);
}

__global__ void __launch_bounds__(kWriteWg) k_decode_write_multi(const DecField* __restrict__ fd,
                                                                 const uint64_t* __restrict__ start, int nf,
                                                                 const uint64_t* __restrict__ off) {
    const uint64_t u = blockIdx.x;
    const int f = field_of(start, nf, u);
    const DecodeArgs a = fd[f].a;
    const SubState s = fd[f].s;
    decode_write_unit<true>(a, s, off + 2 * start[f], off + 2 * u, fd[f].codes, fd[f].sparse, fd[f].sum, u - start[f]);
}

__global__ void k_dec_field_totals(const uint64_t* __restrict__ start, int nf, const uint64_t* __restrict__ off,
                                   uint64_t* __restrict__ tot) {
    const int f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f < nf) tot[f] = off[2 * start[f + 1]] - off[2 * start[f]];
}

// KIND: the tile form of every field in the queue, or -1: each field's own.
template <int KIND, int B>
__global__ void __launch_bounds__(256, (KIND == kRc3x4 || KIND == kRc3x4u || KIND < 0) && B == 8 ? 4 : 1)
    k_recon_multi(const DecField* __restrict__ fd, const uint64_t* __restrict__ start, int nf, uint64_t ntot) {
    const uint64_t wave = blockIdx.x * 4ull + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint64_t nwaves = gridDim.x * 4ull;
    for (uint64_t T = wave; T < ntot; T += nwaves) {
        const int f = field_of(start, nf, T);
        const uint64_t t = T - start[f];
        const ReconArgs ra = fd[f].ra;
        const uint16_t* codes = fd[f].codes;
        const float* sparse = fd[f].sparse;
        float* out = fd[f].out;
        uint32_t* fl = fd[f].flagged;
        uint32_t* nfl = fd[f].nflagged;
        const int kind = KIND < 0 ? fd[f].kind : KIND;
        if (kind == kRc1x4) recon_x4_tile<1, B, true>(t, codes, sparse, out, ra, fl, nfl);
        if (kind == kRc2x4) recon_x4_tile<2, B, true>(t, codes, sparse, out, ra, fl, nfl);
        if (kind == kRc1x4u) recon_x4_tile<1, B, false>(t, codes, sparse, out, ra, fl, nfl);
        if (kind == kRc2x4u) recon_x4_tile<2, B, false>(t, codes, sparse, out, ra, fl, nfl);
        if constexpr (B <= 16) {
            if (kind == kRc3x4) recon_x4_tile<3, B, true>(t, codes, sparse, out, ra, fl, nfl);
            if (kind == kRc3x4u) recon_x4_tile<3, B, false>(t, codes, sparse, out, ra, fl, nfl);
        }
        if (kind == kRc3) recon_3d_tile<B, false>(t, codes, sparse, out, ra, fl, nfl);
        if (kind == kRc2) recon_2d_tile<B, false>(t, codes, sparse, out, ra, fl, nfl);
    }
}

__global__ void __launch_bounds__(256) k_gather_heads(const HeadCopy* __restrict__ hc, uint8_t* __restrict__ dst) {
    const HeadCopy h = hc[blockIdx.x];
    for (uint64_t i = threadIdx.x; i < h.len; i += blockDim.x) dst[h.off + i] = h.src[i];
}

// blockIdx.y: the field.
__global__ void __launch_bounds__(64) k_recon_fallback_multi(int B, const DecField* __restrict__ fd) {
    const DecField& F = fd[blockIdx.y];
    if (F.kind < 0) return;
    recon_fallback_blocks(F.ndim, B, F.codes, F.sparse, F.out, F.ra, F.flagged, F.nflagged,
                          blockIdx.x * (uint64_t)blockDim.x + threadIdx.x, (uint64_t)gridDim.x * blockDim.x);
}

// ------------------------------------------------------------------ launchers

static unsigned grid_for(uint64_t threads, unsigned block) { return (unsigned)((threads + block - 1) / block); }

// Dynamic LDS bytes of the decode tables a kernel keeps in LDS.
static size_t table_lds_bytes(const DecodeArgs& a, bool t16) {
    return t16 ? ((size_t)(1u << kLutBits) + a.n_sub16) * 2 : (size_t)(1u << kLutBits) * 4;
}

// LDS room for deeper compact tables (n_sub16): what is left of a workgroup's
// share of the CU when as many workgroups are resident as its other LDS
// (own_bytes besides the first level) allows.  The tables of codewords of up
// to 16 bits come first; the rest is read in global memory.  (LDS is given
// out in units of 1280 bytes: filling up to a KiB granule instead cost the
// sync pass a workgroup per CU, 0.65 -> 1.0 ms at the 1 GiB field.)
static DecodeArgs with_lds_sub16(DecodeArgs a, size_t own_bytes) {
    a.n_sub16 = 0;
    if (!a.tabs) return a;
    constexpr size_t kCuLds = 160 * 1024, kGranule = 1280;
    const size_t bare = table_lds_bytes(a, true) + own_bytes;
    const size_t share = kCuLds / ((bare + kGranule - 1) / kGranule * kGranule);  // workgroups per CU
    const size_t room = kCuLds / share / kGranule * kGranule - bare;
    a.n_sub16 = (uint32_t)std::min<size_t>(kMaxSub16, room / 2 & ~(size_t)((1u << kSubTabBits) - 1));
    return a;
}

// Lets a kernel take more than the default 64 KiB of dynamic LDS (gfx950
// has 160 KiB per workgroup; the kernels here have no static LDS).  Set once
// per kernel: each call site keeps its own once-flag (kernels of one
// signature share a function type, so a flag per type would skip all but
// the first of them).
static bool set_big_lds(const void* kernel) {
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
        (void)hipGetLastError();  // the launch then reports what does not fit
    return true;
}
#define allow_big_lds(K)                                                                 \
    do {                                                                                 \
        static const bool once_ = set_big_lds(reinterpret_cast<const void*>(&(K)));      \
        (void)once_;                                                                     \
    } while (0)

void launch_decode_sync(const DecodeArgs& a0, SubState s, DecSummary* sum, hipStream_t st) {
    allow_big_lds(k_decode_sync<true>);
    allow_big_lds(k_decode_sync<false>);
    const bool t16 = a0.tabs != nullptr;
    const DecodeArgs a = with_lds_sub16(a0, (size_t)kSyncLdsWords * 4);
    const size_t lds = table_lds_bytes(a, t16) + (size_t)kSyncLdsWords * 4;
    const dim3 grid(grid_for(a.nsub, kSyncStride));
    if (t16)
        hipLaunchKernelGGL(k_decode_sync<true>, grid, dim3(kSyncWg), lds, st, a, s, sum);
    else
        hipLaunchKernelGGL(k_decode_sync<false>, grid, dim3(kSyncWg), lds, st, a, s, sum);
}
void list_stripes(uint64_t units, SubState* s) {
    s->nstripe = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(kMaxStripes, units));
    s->stripe_cap = (units + s->nstripe - 1) / s->nstripe * kSyncWg;
    s->counter_words = kCounterWords;
    s->slot_words = kSlotWords;
}
uint64_t sync_unit_subs() { return kSyncWg; }
static unsigned pass_grid(const SubState& s) {
    return s.nstripe * (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(kPassGrid / s.nstripe, (s.stripe_cap + 255) / 256));
}
void launch_decode_pass(const DecodeArgs& a0, SubState s, uint32_t pass, DecSummary* sum, hipStream_t st) {
    allow_big_lds(k_decode_pass<true>);
    allow_big_lds(k_decode_pass<false>);
    const bool t16 = a0.tabs != nullptr;
    const DecodeArgs a = with_lds_sub16(a0, (size_t)256 * kRowStride * 4);
    const size_t lds = table_lds_bytes(a, t16) + (size_t)256 * kRowStride * 4;
    // persistent workgroups; those past the listed count return at once
    const dim3 grid(pass_grid(s));
    if (t16)
        hipLaunchKernelGGL(k_decode_pass<true>, grid, dim3(256), lds, st, a, s, pass, sum);
    else
        hipLaunchKernelGGL(k_decode_pass<false>, grid, dim3(256), lds, st, a, s, pass, sum);
}
void launch_decode_indexed(const DecodeArgs& a0, const uint64_t* index, uint64_t total_bits, uint16_t* codes,
                           float* sparse, const Recon1D* r1d, DecSummary* sum, hipStream_t st) {
    allow_big_lds((k_decode_indexed<true, false>));
    allow_big_lds((k_decode_indexed<false, false>));
    allow_big_lds((k_decode_indexed<true, true>));
    allow_big_lds((k_decode_indexed<false, true>));
    allow_big_lds((k_decode_indexed_staged<true, false>));
    allow_big_lds((k_decode_indexed_staged<false, false>));
    allow_big_lds((k_decode_indexed_staged<true, true>));
    allow_big_lds((k_decode_indexed_staged<false, true>));
    const bool t16 = a0.tabs != nullptr;
    const DecodeArgs a = with_lds_sub16(a0, (size_t)4 * kIdxStageWords * 4);
    const size_t lds = table_lds_bytes(a, t16) + (size_t)4 * kIdxStageWords * 4;
    const IdxLayout L = idx_layout(a.n);
    const dim3 grid((unsigned)std::max<uint64_t>(1, (L.nseg + 255) / 256));
    const Recon1D r = r1d ? *r1d : Recon1D{};
    // workgroups whose span fits the LDS stage first, then the others through
    // the register-window kernel (which skips the staged ones)
    {
        const DecodeArgs as = with_lds_sub16(a0, (size_t)(kIdxSpanWords + kIdxSpanOver) * 4);
        const size_t lds_s = table_lds_bytes(as, t16) + (size_t)(kIdxSpanWords + kIdxSpanOver) * 4;
#define DS(T, R)                                                                                                    \
    hipLaunchKernelGGL((k_decode_indexed_staged<T, R>), grid, dim3(256), lds_s, st, as, index, L, total_bits, codes, \
                       sparse, r, sum)
        if (r1d) {
            if (t16)
                DS(true, true);
            else
                DS(false, true);
        } else {
            if (t16)
                DS(true, false);
            else
                DS(false, false);
        }
#undef DS
    }
#define DI(T, R) \
    hipLaunchKernelGGL((k_decode_indexed<T, R>), grid, dim3(256), lds, st, a, index, L, total_bits, codes, sparse, r, sum)
    if (r1d) {
        if (t16)
            DI(true, true);
        else
            DI(false, true);
    } else {
        if (t16)
            DI(true, false);
        else
            DI(false, false);
    }
#undef DI
}
void launch_decode_tail(const DecodeArgs& a0, SubState s, uint32_t pass, DecSummary* sum, hipStream_t st) {
    allow_big_lds(k_decode_tail<true>);
    allow_big_lds(k_decode_tail<false>);
    const bool t16 = a0.tabs != nullptr;
    constexpr size_t kOwn = (size_t)kTailWg * (kRowStride * 4 + 2 * 8) + 16;
    const DecodeArgs a = with_lds_sub16(a0, kOwn);
    const size_t lds = table_lds_bytes(a, t16) + kOwn;
    if (t16)
        hipLaunchKernelGGL(k_decode_tail<true>, dim3(1), dim3(kTailWg), lds, st, a, s, pass, sum);
    else
        hipLaunchKernelGGL(k_decode_tail<false>, dim3(1), dim3(kTailWg), lds, st, a, s, pass, sum);
}
void launch_decode_offsets(const SubState& s, uint64_t nsub, uint64_t* off, hipStream_t st, const uint32_t* guard) {
    const uint64_t nu = decode_write_units(nsub);
    if (nu <= kOneOffsets) {
        hipLaunchKernelGGL(k_decode_offsets, dim3(1), dim3(1024), 0, st, s, nsub, (uint32_t)nu, off, guard);
        return;
    }
    hipLaunchKernelGGL(k_decode_sums, dim3(grid_for(nu, 4)), dim3(256), 0, st, s, nsub, nu, off, guard);
    hipLaunchKernelGGL(k_decode_scan, dim3(1), dim3(1024), 0, st, off, nu, guard);
}
void launch_decode_write(const DecodeArgs& a0, SubState s, const uint64_t* off, uint16_t* codes, float* sparse,
                         DecSummary* sum, hipStream_t st, const uint32_t* guard) {
    allow_big_lds(k_decode_write<true>);
    allow_big_lds(k_decode_write<false>);
    const bool t16 = a0.tabs != nullptr;
    const DecodeArgs a = with_lds_sub16(a0, (size_t)kWriteLdsWords * 4);
    const size_t lds = table_lds_bytes(a, t16) + (size_t)kWriteLdsWords * 4;
    const dim3 grid((unsigned)decode_write_units(a.nsub));
    if (t16)
        hipLaunchKernelGGL(k_decode_write<true>, grid, dim3(kWriteWg), lds, st, a, s, off, codes, sparse, sum, guard);
    else
        hipLaunchKernelGGL(k_decode_write<false>, grid, dim3(kWriteWg), lds, st, a, s, off, codes, sparse, sum, guard);
}
void launch_fill_u16(uint16_t* p, uint64_t n, uint16_t v, hipStream_t st) {
    unsigned g = (unsigned)std::min<uint64_t>(grid_for(n, 256), 8192);
    hipLaunchKernelGGL(k_fill_u16, dim3(std::max(g, 1u)), dim3(256), 0, st, p, n, v);
}
void launch_scatter_all_outliers(const uint8_t* outliers, uint64_t n, float* sparse, hipStream_t st) {
    unsigned g = (unsigned)std::min<uint64_t>(grid_for(n, 256), 8192);
    hipLaunchKernelGGL(k_scatter_all, dim3(std::max(g, 1u)), dim3(256), 0, st, outliers, n, sparse);
}

void launch_reconstruct(int ndim, int B, const uint16_t* codes, const float* sparse, float* out, const ReconArgs& a,
                        uint32_t* flagged, uint32_t* nflagged, int grid, hipStream_t st) {
    // four x per lane when rows are whole multiples of 4 and the output is
    // 16-byte aligned (3D keeps B x 4 running values per lane: B <= 16)
    if (a.halo) {
#define RC_PAD(ND, KERN, BB)                                                                                      \
    if (ndim == ND && B == BB) {                                                                                  \
        hipLaunchKernelGGL((KERN<BB, true>), dim3(grid), dim3(256), 0, st, codes, sparse, out, a, flagged, nflagged); \
        return;                                                                                                   \
    }
        RC_PAD(3, k_recon_3d, 8)
        RC_PAD(3, k_recon_3d, 16)
        RC_PAD(3, k_recon_3d, 32)
        RC_PAD(3, k_recon_3d, 64)
        RC_PAD(2, k_recon_2d, 8)
        RC_PAD(2, k_recon_2d, 16)
        RC_PAD(2, k_recon_2d, 32)
        RC_PAD(2, k_recon_2d, 64)
        RC_PAD(1, k_recon_1d, 8)
        RC_PAD(1, k_recon_1d, 16)
        RC_PAD(1, k_recon_1d, 32)
        RC_PAD(1, k_recon_1d, 64)
#undef RC_PAD
        return;
    }
    const int kind = recon_kind(ndim, B, a.d0, codes, out);
    if (kind != kRc2 && kind != kRc3) {
        const uint64_t work = recon_tiles(kind, a);
        const dim3 g4((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((work + 3) / 4, 2048)));
        const bool aln = kind == kRc1x4 || kind == kRc2x4 || kind == kRc3x4;
#define RX4(ND, BB)                                                                                              \
    if (ndim == ND && B == BB) {                                                                                 \
        if (aln)                                                                                                 \
            hipLaunchKernelGGL((k_recon_x4<ND, BB, true>), g4, dim3(256), 0, st, codes, sparse, out, a, flagged,  \
                               nflagged);                                                                        \
        else                                                                                                     \
            hipLaunchKernelGGL((k_recon_x4<ND, BB, false>), g4, dim3(256), 0, st, codes, sparse, out, a, flagged, \
                               nflagged);                                                                        \
        return;                                                                                                  \
    }
        RX4(3, 8)
        RX4(3, 16)
        RX4(2, 8)
        RX4(2, 16)
        RX4(2, 32)
        RX4(2, 64)
        RX4(1, 8)
        RX4(1, 16)
        RX4(1, 32)
        RX4(1, 64)
#undef RX4
    }
#define RC_CASE(ND, KERN, BB)                                                                               \
    if (ndim == ND && B == BB) {                                                                            \
        hipLaunchKernelGGL(KERN<BB>, dim3(grid), dim3(256), 0, st, codes, sparse, out, a, flagged, nflagged); \
        return;                                                                                             \
    }
    RC_CASE(3, k_recon_3d, 8)
    RC_CASE(3, k_recon_3d, 16)
    RC_CASE(3, k_recon_3d, 32)
    RC_CASE(3, k_recon_3d, 64)
    RC_CASE(2, k_recon_2d, 8)
    RC_CASE(2, k_recon_2d, 16)
    RC_CASE(2, k_recon_2d, 32)
    RC_CASE(2, k_recon_2d, 64)
#undef RC_CASE
}

void launch_reconstruct_fallback(int ndim, int B, const uint16_t* codes, const float* sparse, float* out,
                                 const ReconArgs& a, const uint32_t* flagged, const uint32_t* nflagged, hipStream_t st) {
    hipLaunchKernelGGL(k_recon_fallback, dim3(256), dim3(64), 0, st, ndim, B, codes, sparse, out, a, flagged, nflagged);
}

static DecodeArgs compact_probe(uint32_t n_sub16) {
    DecodeArgs probe{};
    probe.tabs = reinterpret_cast<const uint16_t*>(&probe);  // (only tested for null)
    probe.n_sub16 = n_sub16;
    return probe;
}
constexpr size_t kPassRowBytes = (size_t)256 * kRowStride * 4;
uint32_t batch_sub16_in_lds() {
    const DecodeArgs probe = compact_probe(0);
    return std::min({with_lds_sub16(probe, (size_t)kSyncLdsWords * 4).n_sub16,
                     with_lds_sub16(probe, (size_t)kWriteLdsWords * 4).n_sub16,
                     with_lds_sub16(probe, kPassRowBytes).n_sub16});
}

void launch_decode_sync_multi(uint32_t n_sub16, const DecField* fd, const uint64_t* start, int nf, uint64_t nunits,
                              hipStream_t st) {
    allow_big_lds(k_decode_sync_multi);
    if (!nunits) return;
    const size_t lds = table_lds_bytes(compact_probe(n_sub16), true) + (size_t)kSyncLdsWords * 4;
    hipLaunchKernelGGL(k_decode_sync_multi, dim3((unsigned)nunits), dim3(kSyncWg), lds, st, fd, start, nf);
}
void launch_decode_pass_multi(uint32_t n_sub16, const DecField* fd, const uint64_t* start, int nf, uint64_t nunits,
                              uint32_t pass, hipStream_t st) {
    allow_big_lds(k_decode_pass_multi);
    if (!nunits) return;
    const size_t lds = table_lds_bytes(compact_probe(n_sub16), true) + kPassRowBytes;
    hipLaunchKernelGGL(k_decode_pass_multi, dim3((unsigned)nunits), dim3(256), lds, st, fd, start, nf, pass);
}
void launch_decode_offsets_multi(const DecField* fd, const uint64_t* start, int nf, uint64_t nunits, uint64_t* off,
                                 hipStream_t st) {
    if (nunits)
        hipLaunchKernelGGL(k_decode_sums_multi, dim3(grid_for(nunits, 4)), dim3(256), 0, st, fd, start, nf, off);
    hipLaunchKernelGGL(k_decode_scan, dim3(1), dim3(1024), 0, st, off, nunits, (const uint32_t*)nullptr);
}
void launch_decode_write_multi(uint32_t n_sub16, const DecField* fd, const uint64_t* start, int nf, uint64_t nunits,
                               const uint64_t* off, hipStream_t st) {
    allow_big_lds(k_decode_write_multi);
    if (!nunits) return;
    const size_t lds = table_lds_bytes(compact_probe(n_sub16), true) + (size_t)kWriteLdsWords * 4;
    hipLaunchKernelGGL(k_decode_write_multi, dim3((unsigned)nunits), dim3(kWriteWg), lds, st, fd, start, nf, off);
}
void launch_dec_field_totals(const uint64_t* start, int nf, const uint64_t* off, uint64_t* tot, hipStream_t st) {
    if (nf > 0)
        hipLaunchKernelGGL(k_dec_field_totals, dim3(grid_for((uint64_t)nf, 256)), dim3(256), 0, st, start, nf, off, tot);
}
int recon_kind_ndim(int kind) {
    switch (kind) {
        case kRc1x4: case kRc1x4u: return 1;
        case kRc2: case kRc2x4: case kRc2x4u: return 2;
        default: return 3;
    }
}
int recon_kind(int ndim, int B, uint64_t d0, const void* codes, const void* out) {
    // four x per lane unless a 3D tile's B x 4 running values per lane would
    // not fit (B > 16); vector loads and stores when rows are whole multiples
    // of 4 and codes / output are 8- / 16-byte aligned
    if (ndim == 3 && B > 16) return kRc3;
    // under 128 wide the 4-wide tiles' 256 columns are half empty, and a row
    // costs a wavefront four elements' instructions: 64 columns, one element
    // a lane (25 x 25 x 26: stage 47 -> 26 us)
    if (ndim > 1 && d0 < 128) return ndim == 2 ? kRc2 : kRc3;
    const bool aln = d0 % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(codes) & 7) == 0;
    if (ndim == 1) return aln ? kRc1x4 : kRc1x4u;
    if (ndim == 2) return aln ? kRc2x4 : kRc2x4u;
    return aln ? kRc3x4 : kRc3x4u;
}
uint64_t recon_tiles(int kind, const ReconArgs& a) {
    const bool x4 = kind != kRc2 && kind != kRc3;
    const int nd = recon_kind_ndim(kind);
    const uint64_t tx = x4 ? (a.d0 + 255) / 256 : a.ntiles_x;
    return tx * (nd >= 2 ? a.ntiles_y : 1) * (nd >= 3 ? a.ntiles_z : 1);
}
void launch_reconstruct_multi(int kind, int B, const DecField* fd, const uint64_t* start, int nf, uint64_t ntiles,
                              hipStream_t st) {
    if (!ntiles) return;
    const dim3 grid((unsigned)std::max<uint64_t>(1, std::min<uint64_t>((ntiles + 3) / 4, 2048)));
#define RM(K, BB)                                                                                \
    if (kind == K && B == BB) {                                                                  \
        hipLaunchKernelGGL((k_recon_multi<K, BB>), grid, dim3(256), 0, st, fd, start, nf, ntiles); \
        return;                                                                                  \
    }
#define RM_B(BB) RM(-1, BB) RM(kRc1x4, BB) RM(kRc1x4u, BB) RM(kRc2, BB) RM(kRc2x4, BB) RM(kRc2x4u, BB) RM(kRc3, BB)
    RM_B(8) RM_B(16) RM_B(32) RM_B(64)
    RM(kRc3x4, 8) RM(kRc3x4, 16) RM(kRc3x4u, 8) RM(kRc3x4u, 16)
#undef RM_B
#undef RM
}
uint64_t decode_sync_units(uint64_t nsub) { return (nsub + kSyncStride - 1) / kSyncStride; }
uint64_t decode_write_units(uint64_t nsub) { return (nsub + kWriteWg - 1) / kWriteWg; }
void launch_gather_heads(const HeadCopy* hc, int n, uint8_t* dst, hipStream_t st) {
    if (n > 0) hipLaunchKernelGGL(k_gather_heads, dim3((unsigned)n), dim3(256), 0, st, hc, dst);
}
void launch_reconstruct_fallback_multi(int B, const DecField* fd, int nf, hipStream_t st) {
    if (nf > 0) hipLaunchKernelGGL(k_recon_fallback_multi, dim3(16, (unsigned)nf), dim3(64), 0, st, B, fd);
}

}  // namespace vsz
