// Host tables of the string form (strings.hpp): strings, single replacements and the lists that let each
// kernel walk its determinants or strings without searching.
#include <algorithm>
#include <bit>
#include <cstdlib>

#include "strings.hpp"

namespace xmvb_amd {
namespace {

// parity of replacing l by q in a string (q unoccupied, or q == l)
bool odd_replacement(uint32_t mask, int l, int q) {
    const int lo = std::min(l, q), hi = std::max(l, q);
    const uint32_t between = ((1u << hi) - 1) & ~((2u << lo) - 1);
    return hi > lo && (std::popcount(mask & between) & 1);
}

StringTables::Space make_space(int n, int m, const std::vector<uint16_t>& rank) {
    StringTables::Space s;
    s.m = m;
    s.noff = m * (n - m);
    s.J = s.noff + m;
    for (uint32_t x = 0; x < (1u << n); ++x)
        if (std::popcount(x) == m) s.mask.push_back(x);
    s.N = (int)s.mask.size();
    s.e1.reserve((size_t)s.N * s.J);
    for (const uint32_t x : s.mask) {
        for (int l = 0; l < n; ++l)
            for (int q = 0; q < n; ++q)
                if ((x >> l & 1) && !(x >> q & 1))
                    s.e1.push_back((uint32_t)rank[x ^ (1u << l) ^ (1u << q)] | (uint32_t)(q * n + l) << 16 |
                                   (odd_replacement(x, l, q) ? 1u << 31 : 0u));
        for (int l = 0; l < n; ++l)
            if (x >> l & 1) s.e1.push_back((uint32_t)rank[x] | (uint32_t)(l * n + l) << 16);
    }
    return s;
}

void csr(int n, const std::vector<int>& key, std::vector<int>& off, std::vector<int>& items) {
    off.assign(n + 1, 0);
    for (const int k : key) ++off[k + 1];
    for (int k = 0; k < n; ++k) off[k + 1] += off[k];
    items.resize(key.size());
    auto at = off;
    for (int i = 0; i < (int)key.size(); ++i) items[at[key[i]]++] = i;
}

}  // namespace

StringTables build_string_tables(int n, int n_alpha, int n_beta, int n_det, const uint64_t* amask, const int* det_a,
                                 const uint64_t* bmask, const int* det_b, const long long* off, const int* ts,
                                 const double* tc, const std::vector<int>& flip) {
    StringTables t;
    t.n = n;
    if (n > 14 || n_alpha < 1 || n_beta < 1 || n_alpha > 7 || n_beta > 7 || n_alpha >= n ||
        n_beta >= n || n_det < kStringDetsMin || n_det > kStringDetsMax)
        return t;
    t.rank.assign(1u << n, 0);
    {
        std::vector<int> seen(n + 1, 0);
        for (uint32_t x = 0; x < (1u << n); ++x) t.rank[x] = (uint16_t)seen[std::popcount(x)]++;
    }
    t.a = make_space(n, n_alpha, t.rank);
    t.b = make_space(n, n_beta, t.rank);
    // f and sigma lie over the determinant matrices
    if ((long long)t.a.N * t.b.N > (long long)n_det * n_det) return t;
    t.arank.resize(n_det);
    t.brank.resize(n_det);
    for (int d = 0; d < n_det; ++d) {
        t.arank[d] = t.rank[(uint32_t)amask[det_a[d]]];
        t.brank[d] = t.rank[(uint32_t)bmask[det_b[d]]];
    }
    csr(t.a.N, t.arank, t.aoff, t.adet);
    csr(t.b.N, t.brank, t.boff, t.bdet);
    for (int s = 0; s < t.a.N; ++s)  // each determinant once
        for (int i = t.aoff[s]; i < t.aoff[s + 1]; ++i)
            for (int k = i + 1; k < t.aoff[s + 1]; ++k)
                if (t.brank[t.adet[i]] == t.brank[t.adet[k]]) return t;

    // exchange of the spins: the same term list up to one common sign for every determinant
    if (n_alpha == n_beta) {
        int sign = 0;
        bool ok = true;
        for (int d = 0; d < n_det && ok; ++d) {
            int f = -1;
            for (int i = t.aoff[t.brank[d]]; i < t.aoff[t.brank[d] + 1]; ++i)
                if (t.brank[t.adet[i]] == t.arank[d]) f = t.adet[i];
            ok = f >= 0 && off[d + 1] - off[d] == off[f + 1] - off[f];
            for (long long k = 0; ok && k < off[d + 1] - off[d]; ++k) {
                const double x = tc[off[d] + k], y = tc[off[f] + k];
                ok = ts[off[d] + k] == ts[off[f] + k] && (x == y || x == -y);
                if (ok && x != 0.0) {
                    const int s = x == y ? 1 : -1;
                    if (sign == 0) sign = s;
                    ok = s == sign;
                }
            }
        }
        t.sym = !ok ? 0 : sign < 0 ? -1 : 1;
    }

    // sigma rows: x = a with l replaced by q, reached from a = x with q replaced by l
    const int n2 = n * n;
    t.soff.push_back(0);
    for (int x = 0; x < t.a.N; ++x) {
        auto push = [&](int a, uint32_t pair, uint32_t odd) {
            for (int i = t.aoff[a]; i < t.aoff[a + 1]; ++i) t.slink.push_back({(uint32_t)t.adet[i], pair | odd});
        };
        for (int j = 0; j < t.a.noff; ++j) {
            const uint32_t e = t.a.e1[(size_t)x * t.a.J + j];
            const int from = (int)(e >> 16 & 0xff), l = from / n, q = from % n;
            push((int)(e & 0xffff), (uint32_t)(q * n + l), e & (1u << 31));
        }
        push(x, (uint32_t)n2, 0u);
        t.soff.push_back((int)t.slink.size());
    }
    // (q, l) -> determinants
    std::vector<std::vector<StringLink>> per(n2);
    for (int d = 0; d < n_det; ++d)
        for (int j = 0; j < t.a.J; ++j) {
            const uint32_t e = t.a.e1[(size_t)t.arank[d] * t.a.J + j];
            per[e >> 16 & 0xff].push_back({(uint32_t)d, (e & 0xffff) | (e & (1u << 31))});
        }
    t.goff.push_back(0);
    size_t longest = 0;
    for (auto& v : per) {
        longest = std::max(longest, v.size());
        t.glink.insert(t.glink.end(), v.begin(), v.end());
        t.goff.push_back((int)t.glink.size());
    }
    t.gchunks = (int)((longest + 63) / 64);
    // response sum: one beta electron fewer
    for (uint32_t w = 0; w < (1u << n); ++w) {
        if (std::popcount(w) != n_beta - 1) continue;
        for (int q = 0; q < 16; ++q) {
            const bool free = q < n && !(w >> q & 1);
            const int odd = free ? std::popcount(w & ((1u << q) - 1)) & 1 : 0;
            t.wtab.push_back((uint16_t)((free ? t.rank[w | 1u << q] : t.b.N) | odd << 15));
        }
        ++t.nw;
    }
    // same-spin densities: double replacements
    const int nc = n * (n - 1) / 2;
    auto doubles = [&](const StringTables::Space& s, const std::vector<int>& rank_of, std::vector<uint32_t>& out, int& nq,
                       std::vector<int>& off2, std::vector<StringLink>& link2) {
        auto below = [](uint32_t v, int k) { return std::popcount(v & ((1u << k) - 1)); };
        std::vector<std::vector<StringLink>> dets(nc);
        nq = (n - s.m + 2) * (n - s.m + 1) / 2;
        for (const uint32_t m : s.mask)
            for (int l2 = 1; l2 < n; ++l2)
                for (int l = 0; l < l2; ++l) {
                    if (!(m >> l & 1) || !(m >> l2 & 1)) continue;
                    const uint32_t rest = m ^ 1u << l ^ 1u << l2;
                    for (int q2 = 1; q2 < n; ++q2)
                        for (int q = 0; q < q2; ++q) {
                            if ((rest >> q & 1) || (rest >> q2 & 1)) continue;
                            const int odd = below(m, l) + below(m ^ 1u << l, l2) + below(rest, q2) + below(rest | 1u << q2, q);
                            out.push_back((uint32_t)t.rank[rest | 1u << q | 1u << q2] |
                                          (uint32_t)(q2 * (q2 - 1) / 2 + q) << 12 | (odd & 1 ? 1u << 31 : 0u));
                        }
                }
        for (int d = 0; d < n_det; ++d) {
            uint32_t place = 0;
            for (int l2 = 1; l2 < n; ++l2)
                for (int l = 0; l < l2; ++l)
                    if ((s.mask[rank_of[d]] >> l & 1) && (s.mask[rank_of[d]] >> l2 & 1))
                        dets[l2 * (l2 - 1) / 2 + l].push_back({(uint32_t)d, place++});
        }
        off2.push_back(0);
        for (const auto& v : dets) {
            link2.insert(link2.end(), v.begin(), v.end());
            off2.push_back((int)link2.size());
            t.wchunks = std::max(t.wchunks, (int)((v.size() + 63) / 64));
        }
    };
    doubles(t.b, t.brank, t.e2b, t.nq_b, t.w2off_b, t.w2link_b);
    doubles(t.a, t.arank, t.e2a, t.nq_a, t.w2off_a, t.w2link_a);
    // determinant pairs: one determinant of each spin-flip couple against its own and the earlier couples
    const int segment = n_det > 1000 ? 4 * kStringPairSegment : kStringPairSegment;
    std::vector<int> heads;
    for (int d = 0; d < n_det; ++d)
        if (flip.empty() || flip[d] >= d) heads.push_back(d);
    const int lanes = flip.empty() ? 16 : 8;  // couples per block of sixteen positions
    t.order.assign((heads.size() + lanes - 1) / lanes * 16, StringDet{-1, 0, 0, 0});
    for (int k = 0; k < (int)heads.size(); ++k) {
        const int d = heads[k], f = flip.empty() ? d : flip[d], at = k / lanes * 16 + k % lanes;
        t.order[at] = {d, t.arank[d], t.brank[d], f};
        if (f != d) t.order[at + 8] = {f, t.arank[f], t.brank[f], d};
        const int end = (k / lanes + 1) * 16;
        for (int b = 0; b < end; b += segment) t.pitem.push_back({d, b, std::min(end, b + segment), k});
    }
    // and over the alpha strings
    std::vector<std::vector<uint32_t>> al(n2);
    for (int x = 0; x < t.a.N; ++x)
        for (int j = 0; j < t.a.J; ++j) al[t.a.e1[(size_t)x * t.a.J + j] >> 16 & 0xff].push_back((uint32_t)(x * t.a.J + j));
    for (auto& v : al) t.ak = std::max(t.ak, (int)v.size());
    t.alist.assign((size_t)t.ak * n2, ~0u);
    for (int p = 0; p < n2; ++p)
        for (size_t k = 0; k < al[p].size(); ++k) t.alist[k * n2 + p] = al[p][k];
    t.enabled = true;
    return t;
}

}  // namespace xmvb_amd
