// Evaluation over the strings of the active space ("string form"), see strings.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <vector>

namespace xmvb_amd {

// All strings of m electrons in n orbitals, in ascending mask order, with their single replacements:
// e1[x * J + j], j < noff: l -> q with q unoccupied, then the m occupied orbitals (q == l). An entry
// packs the rank of the resulting string (bits 0-15), q n + l (16-23) and the parity (31).
struct StringSpace {
    int m, N, noff, J;
    const uint32_t* mask;
    const uint32_t* e1;
};

// One determinant reached from a string row: determinant, and packed (rank or orbital pair, parity).
struct StringLink {
    uint32_t det;
    uint32_t to;  // bits 0-15: rank of the replaced string, or q n + l (n^2: no replacement); 31: parity
};

// A determinant (negative: padding) with its string ranks and its spin-flip partner (itself without one).
struct StringDet {
    int det, a, b, flip;
};

// Determinant pairs {order[begin..end), det}, those with order_couple(position) <= couple.
struct StringPairItem {
    int det, begin, end, couple;
};

// Couple of a position of the order: blocks of sixteen hold one determinant of each of eight couples, then
// their partners, so that either half runs along consecutive strings.
__host__ __device__ inline int order_couple(int position, bool flip) {
    return flip ? 8 * (position >> 4) + (position & 7) : position;
}

// Topology tables of the string form (device pointers).
struct StringTopo {
    int enabled;  // 0: this topology takes the pair kernels
    int sym;      // +-1: exchanging the spins multiplies every determinant coefficient by it; 0: no such sign
    StringSpace a, b;
    const uint16_t* rank;              // mask -> rank among the masks of the same electron count
    const int *arank, *brank;          // determinant -> string ranks
    const int *aoff, *adet;            // alpha string -> determinants
    const int *boff, *bdet;            // beta string -> determinants
    const int* soff;                   // alpha string -> determinants one alpha replacement away
    const StringLink* slink;
    const int* goff;                   // (q, l) -> determinants whose alpha string allows l -> q
    const StringLink* glink;
    int gchunks;                       // chunks of 64 links of the longest (q, l) list
    // determinant pairs: the determinants in order (order_couple) and the wavefront items of k_string_pairs
    const StringDet* order;
    const StringPairItem* pitem;
    int npitem;
    // alpha strings for the same, as offsets x * J + j per (q, l): [ak][n^2], ~0 past the end
    const uint32_t* alist;
    int ak;
    // strings of one beta electron fewer, [nw][16]: rank of the string with orbital q added (bits 0-11; N
    // where q is occupied or past n) and the parity of q's place (15)
    const uint16_t* wtab;
    // double replacements l < l2 -> q < q2 of every string (q, q2 may be l, l2), [N][pairs l l2][nq]: rank
    // (0-11), compound index of (q, q2) (12-18), parity (31)
    const uint32_t *e2a, *e2b;
    // (l, l2) -> determinants whose beta (alpha) string holds both, and the place of l l2 among its pairs
    const int *w2off_b, *w2off_a;
    const StringLink *w2link_b, *w2link_a;
    int nw, nq_a, nq_b, wchunks;
};

// Host image of the tables, built once per pool.
struct StringTables {
    bool enabled = false;
    int sym = 0, n = 0;
    struct Space {
        int m = 0, N = 0, noff = 0, J = 0;
        std::vector<uint32_t> mask, e1;
    } a, b;
    std::vector<uint16_t> rank;
    std::vector<int> arank, brank, aoff, adet, boff, bdet, soff, goff;
    std::vector<StringLink> slink, glink;
    std::vector<uint32_t> alist, e2a, e2b;
    std::vector<uint16_t> wtab;
    std::vector<StringDet> order;
    std::vector<StringPairItem> pitem;
    std::vector<int> w2off_a, w2off_b;
    std::vector<StringLink> w2link_a, w2link_b;
    int gchunks = 0, ak = 0, nw = 0, nq_a = 0, nq_b = 0, wchunks = 0;
};

StringTables build_string_tables(int n, int n_alpha, int n_beta, int n_det, const uint64_t* amask, const int* det_a,
                                 const uint64_t* bmask, const int* det_b, const long long* off, const int* ts,
                                 const double* tc, const std::vector<int>& flip);

// Arrays of one slot. The determinant matrices are dead once the structure matrices are formed, so
// f and sigma (with C M before it) take their place.
struct StringWork {
    double *Sinv, *ht;   // S_act^-1, S_act^-1 h_act (n x n, row-major)
    double *U, *gt;      // S_act^-1 on one, on both sides of the packed kernel: [q n + l][pair], [q n + l][q2 n + l2]
    double *Ma, *Mb;     // minors of S_act over all string pairs
    double *Ja, *Jb;     // sum over the occupied l2 of gt[q n + l][l2 l2], per string
    double *Ha, *Hb;     // same-spin Hamiltonian in the dual frame, [x][a]
    unsigned char *neara, *nearb;  // string pairs: conditioning of the overlap block, [y][x] for x <= y (k_string_condition)
    double *Ka, *Kb;     // same-spin Hamiltonian between strings; during the forward, over gpart and on
    double *gpart, *wpart, *zpart;
    double *gs, *hb, *V, *W2, *Zt;
    double *Fa, *Fb;     // ht + Coulomb - exchange of each string, [x][ql]
};

// Where the string form is the faster one: from kStringWork on of the pair kernels' leading work, n_det^2 (m_a m_b)^2
// over all problems of the launch (of one problem for pinned shapes, whose form may not depend on the batch).
// Both forms in one build, whole calls of 100 basis functions in us, string form / pair kernels, by that work: 126 determinants
// (5 + 4 electrons) x 16 1.0e8 837/702, x 64 4.1e8 1501/1607; 210 (6 + 4) x 1 2.5e7 1137/903, x 8 2.0e8 1284/1364; 252
// (5 + 5) x 1 4.0e7 540/518, x 4 1.6e8 676/628, x 8 3.2e8 721/783, x 64 2.5e9 1740/2700; 400 on 20 strings (3 + 3) x 8
// 1.0e8 1393/1317, x 16 2.1e8 1470/1490, x 64 8.3e8 2279/2576; 462 (6 + 5) x 1 1.9e8 1581/1465, x 4 7.7e8 1837/2796; 924
// (6 + 6) x 1 1.1e9 1340/1992. Not measured, and on the pair kernels: spaces of fewer than kStringDetsMin or more
// than kStringDetsMax determinants.
constexpr double kStringWork = 3.0e8;
constexpr int kStringDetsMin = 100, kStringDetsMax = 4096;
constexpr int kStringRowsZ = 8;         // rows of f and sigma per workgroup of the response sum
constexpr int kStringPairSegment = 128; // determinants per wavefront of k_string_pairs (512 in large spaces)
// Pairs left to the list kernels, energy and gradient: those whose regular inverse form loses digits, so that
// both forms give the same result whatever the slot, the batch or the limits choose. The inverse form of the
// gradient cancels terms of size |S_de| max|X^-1|^3 down to S_de's own size. Over 1,477 problems of 9 to 14 orbitals
// the relative difference of the two forms' gradients stayed below 1e-17 times the sum of that over the pairs of
// the strings, divided by the number of determinants (median 8e-20), and reached 8.8e-6 without a list. This
// limit per pair (divided likewise) keeps the sum below 7e6; the difference then stayed below 1.8e-10, with a median
// of 2 pairs listed at 10 orbitals and 20 at 12 to 14. A block the lane kernels keep (condition below
// kLaneConditionDefault) is never listed; one that may be rank deficient (above kLaneConditionMax) always is.
constexpr double kStringListError = 1.0e5;
// Above this many listed pairs a slot stays on the pair kernels. A pair costs 2 us in one problem of 12 orbitals (so all of
// them 0.5 of the 0.65 ms that the strings save there), 6 in one of 14, 0.3 in eight of 12.
constexpr int kStringListMax = 256;
constexpr int kStringListRows = 32;     // workgroups (partial rows) of the listed pairs' response
// Largest |S_act^-1| element (orbitals of unit norm) for which a slot takes the string form. Separate orbitals have 1 to
// 3; drawn together to 15, 12 orbitals, the gradients of the forms agree to 2.3e-12. Not measured beyond.
constexpr double kStringInverseLimit = 16.0;

struct SlotDesc;
struct TopoDesc;

// layout of a slot's StringWork in one block of doubles (base null: only counted); returns their number
std::size_t string_work_carve(const TopoDesc& topo, double* base, StringWork& w);

// S_act^-1 and the route of each slot (FLAG_STRINGS); after the active matrices
void launch_string_frame(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo);
// minors of S_act and the pairs left to the list kernels (flags per work item of the lane kernels, FLAG_NEAR)
void launch_string_minors(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo);
// transformed integrals and the same-spin Hamiltonian
void launch_string_integrals(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo);
// determinant matrices (SlotDesc::Hdet, Sdet)
void launch_string_forward(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo);
// adjoints of the packed kernel, S_act and h_act into SlotDesc::dsum, without the listed pairs
void launch_string_backward(hipStream_t st, const SlotDesc* slots, unsigned z, const TopoDesc& topo);
hipError_t configure_strings();

}  // namespace xmvb_amd
