// The Huffman decode tables built on the device from an archive's tree.
//
//   k_decode_tables  one workgroup per tree (unpad_tree_*, src/huffman.hh:
//                    498-559, :561-643): the node arrays become child words
//                    in LDS, then every table entry walks its own bits
//
// Compact (16-bit) tables only, of trees of at most kMaxTreeNodes nodes whose
// symbols are below 4096 and whose nodes are numbered parents first, as the
// reference's and this library's trees are.  Any other tree (or a damaged
// one) sets the status word: the decode kernels then do nothing, and the host
// builds the 32-bit tables or reports what is wrong.
#include "common.hpp"
#include "kernels.hpp"

namespace vsz {

namespace {

constexpr uint32_t kThreads = 1024;
constexpr uint32_t kNodesPer = (kMaxTreeNodes + kThreads - 1) / kThreads;
constexpr uint32_t kLeaf = 0x8000u;  // child word halves: kLeaf | symbol, or a node

template <typename T>
__device__ __forceinline__ T load_any(const uint8_t* p) {  // any alignment
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

}  // namespace

// What bounds it is latency: 13 rounds of dependent LDS reads for the first
// level and 4 for each deeper one (about 5 at 3,500 symbols), after one round
// trip for the nodes.  The host took 60 to 80 us for such a tree, plus a
// 128 KiB copy down and the tables' copy up; one workgroup takes 10 to 27 us, and
// a batch's trees run side by side.
__global__ void __launch_bounds__(kThreads) k_decode_tables(TableJob one, const TableJob* __restrict__ many) {
    __shared__ uint32_t child[kMaxTreeNodes + 1];  // left | right << 16
    __shared__ uint16_t node_word[kMaxTreeNodes + 1];
    __shared__ uint32_t seen[(kMaxTreeNodes + 32) / 32];
    __shared__ uint32_t bad, internal, nnext;
    // nodes whose tables this level fills and the next one's (node_word's
    // space, free once the child words are there)
    uint16_t* front = node_word;
    uint16_t* next = node_word + kMaxSubTabs;
    static_assert(2 * kMaxSubTabs <= kMaxTreeNodes + 1, "both lists fit");
    const TableJob job = many ? many[blockIdx.x] : one;
    const uint32_t t = threadIdx.x, nc = job.nodes;
    if (nc == 0) return;  // (a batch's field without a tree to build)
    for (uint32_t i = t; i < (kMaxTreeNodes + 32) / 32; i += kThreads) seen[i] = 0;
    if (t == 0) bad = internal = nnext = 0;

    // the node arrays: [u8 0][left][right][symbol u32][leaf u8], all of a
    // thread's loads in flight together
    const uint32_t w = nc <= 256 ? 1 : 2;
    const uint8_t* L = job.huff + 9;
    const uint8_t* R = L + (size_t)nc * w;
    const uint8_t* C = R + (size_t)nc * w;
    const uint8_t* T = C + (size_t)nc * 4;
    uint32_t l[kNodesPer], r[kNodesPer], c[kNodesPer], leaf[kNodesPer];
#pragma unroll
    for (uint32_t m = 0; m < kNodesPer; m++) {
        const uint32_t i = t + m * kThreads;
        if (i < nc) {
            l[m] = w == 1 ? L[i] : load_any<uint16_t>(L + 2 * i);
            r[m] = w == 1 ? R[i] : load_any<uint16_t>(R + 2 * i);
            c[m] = load_any<uint32_t>(C + 4 * (size_t)i);
            leaf[m] = T[i];
        }
    }
    lds_sync();
    bool wrong = false;
#pragma unroll
    for (uint32_t m = 0; m < kNodesPer; m++) {
        const uint32_t i = t + m * kThreads;
        if (i < nc) {
            // (the root of more than 256 nodes is internal whatever its mark
            // says, src/huffman.hh:602)
            if (i == 0 && nc > 256) leaf[m] = 0;
            wrong |= leaf[m] != 0 && (c[m] >= 4096 || i == 0);
            node_word[i] = (uint16_t)(leaf[m] ? kLeaf | (c[m] & 0xFFF) : i);
        }
    }
    lds_sync();
    // every node but the root is the child of one node before it: a full
    // binary tree, all of it reachable
    uint32_t ni = 0;
#pragma unroll
    for (uint32_t m = 0; m < kNodesPer; m++) {
        const uint32_t i = t + m * kThreads;
        if (i < nc && !leaf[m]) {
            ni++;
            const bool ok = l[m] > i && l[m] < nc && r[m] > i && r[m] < nc && l[m] != r[m];
            wrong |= !ok;
            if (ok) {
                wrong |= (atomicOr(&seen[l[m] / 32], 1u << (l[m] % 32)) >> (l[m] % 32)) & 1;
                wrong |= (atomicOr(&seen[r[m] / 32], 1u << (r[m] % 32)) >> (r[m] % 32)) & 1;
                child[i] = (uint32_t)node_word[l[m]] | ((uint32_t)node_word[r[m]] << 16);
            }
        }
    }
    if (ni) atomicAdd(&internal, ni);
    if (wrong) atomicOr(&bad, 1u);
    lds_sync();
    bool fail = bad || 2 * internal + 1 != nc;  // (uniform)

    uint32_t tables = 0;
    if (!fail) {
        // first level: the first codeword of each 12-bit pattern (lut16), and
        // all the codewords that lie in it whole (lut_count, ends); a pattern
        // that is no whole codeword gets a table
        uint16_t* lut_count = job.tabs;
        uint16_t* lut16 = job.tabs + kTabLut;
        uint16_t* ends = job.tabs + kTabEnds;
        uint16_t* sub16 = job.tabs + kTabDeep;
#pragma unroll
        for (uint32_t q = 0; q < (1u << kLutBits) / kThreads; q++) {
            const uint32_t idx = t + q * kThreads;
            uint32_t node = 0, first = 0, end = 0, n = 0, z = 0, at_end = 0;
#pragma unroll
            for (uint32_t b = 0; b < (uint32_t)kLutBits; b++) {
                const uint32_t cw = child[node];
                const uint32_t k = (idx >> (kLutBits - 1 - b)) & 1 ? cw >> 16 : cw & 0xFFFF;
                const bool at = (k & kLeaf) != 0;
                if (at && n == 0) first = ((b + 1) << 12) | (k & 0xFFF);
                n += at;
                z += at && (k & 0xFFF) == 0;
                end = at ? b + 1 : end;
                at_end |= (uint32_t)at << (b + 1);
                node = at ? 0 : k;
            }
            uint32_t e16 = first, ec = (end << 12) | (z << 4) | n;
            if (n == 0) {
                const uint32_t k = atomicAdd(&nnext, 1u);
                if (k < job.cap) front[k] = (uint16_t)node;
                e16 = ec = k;
            }
            lut16[idx] = (uint16_t)e16;
            lut_count[idx] = (uint16_t)ec;
            ends[idx] = (uint16_t)(at_end | (z != 0));
        }
        lds_sync();
        uint32_t nf = nnext;
        // deeper levels: nodes `depth` bits deep, 16 entries each
        for (uint32_t depth = kLutBits; nf != 0; depth += kSubTabBits) {
            // (codewords of more than 64 bits, or more tables than the entries number)
            if (depth + kSubTabBits > 64 || tables + nf > job.cap) {
                fail = true;
                break;
            }
            lds_sync();  // nnext has been read
            if (t == 0) nnext = 0;
            lds_sync();
            for (uint32_t e = t; e < nf << kSubTabBits; e += kThreads) {
                uint32_t node = front[e >> kSubTabBits], out = 0;
#pragma unroll
                for (uint32_t b = 0; b < (uint32_t)kSubTabBits; b++) {
                    if (out == 0) {
                        const uint32_t cw = child[node];
                        const uint32_t k = (e >> (kSubTabBits - 1 - b)) & 1 ? cw >> 16 : cw & 0xFFFF;
                        if (k & kLeaf)
                            out = ((b + 1) << 12) | (k & 0xFFF);
                        else
                            node = k;
                    }
                }
                if (out == 0) {
                    const uint32_t k = atomicAdd(&nnext, 1u);
                    if (k < kMaxSubTabs) next[k] = (uint16_t)node;
                    out = tables + nf + k;  // (past the cap: the next round fails)
                }
                sub16[((size_t)tables << kSubTabBits) + e] = (uint16_t)out;
            }
            lds_sync();
            tables += nf;
            nf = nnext;
            uint16_t* s = front;
            front = next;
            next = s;
        }
    }
    if (t == 0) {
        job.meta->status = fail ? 1u : 0u;
        job.meta->n_sub16 = fail ? 0u : tables << kSubTabBits;
        if (fail && job.hold)
            for (uint32_t p = 0; p < 3; p++) job.hold[list_hold(p)] = 1u;
    }
}

void launch_decode_tables(const TableJob& job, hipStream_t st) {
    hipLaunchKernelGGL(k_decode_tables, dim3(1), dim3(kThreads), 0, st, job, (const TableJob*)nullptr);
}
void launch_decode_tables_multi(const TableJob* jobs, int n, hipStream_t st) {
    if (n > 0) hipLaunchKernelGGL(k_decode_tables, dim3((unsigned)n), dim3(kThreads), 0, st, TableJob{}, jobs);
}

}  // namespace vsz
