// The diagonal Levenshtein decision (lvdist.h) against the dynamic program:
// every pair of short strings over small alphabets, and random pairs with
// lengths around the word edges and distances around the threshold.
#include <algorithm>
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "../../immunodbscan_amd/csrc/lvdist.h"

static long fails = 0, checked = 0;

static int lev(const std::string &a, const std::string &b)
{
    std::vector<int> r(b.size() + 1);
    for (size_t j = 0; j <= b.size(); ++j) r[j] = (int)j;
    for (size_t i = 1; i <= a.size(); ++i) {
        int diag = r[0];
        r[0] = (int)i;
        for (size_t j = 1; j <= b.size(); ++j) {
            const int up = r[j];
            r[j] = std::min({up + 1, r[j - 1] + 1, diag + (a[i - 1] != b[j - 1])});
            diag = up;
        }
    }
    return r[b.size()];
}

template <int NP, int W, int T>
static void one(const std::string &a, const std::string &b, int t, int d, uint32_t junk)
{
    // bits past a row's end hold junk: they must not matter
    uint32_t x[NP * W], y[NP * W];
    for (int p = 0; p < NP; ++p)
        for (int w = 0; w < W; ++w) {
            x[p * W + w] = junk * (p + 3) ^ (junk >> w);
            y[p * W + w] = junk * (p + 7) ^ (junk << w);
            for (int i = 0; i < 32; ++i) {
                const size_t k = 32 * w + i;
                if (k < a.size()) x[p * W + w] = (x[p * W + w] & ~(1u << i)) | ((uint32_t)(a[k] >> p & 1) << i);
                if (k < b.size()) y[p * W + w] = (y[p * W + w] & ~(1u << i)) | ((uint32_t)(b[k] >> p & 1) << i);
            }
        }
    ++checked;
    if (idb_lv_within<NP, W, T>(x, y, (int)a.size(), (int)b.size(), t) != (d <= t))
        if (++fails < 6) std::printf("NP %d W %d T %d t %d: %zu %zu lev %d\n", NP, W, T, t, a.size(), b.size(), d);
}

// rows of equal length: a decision must be the right one
static long decided = 0, asked = 0;
template <int NP, int W, int T>
static void equal(const std::string &a, const std::string &b, int t, int d, uint32_t junk)
{
    uint32_t x[NP * W], y[NP * W];
    for (int p = 0; p < NP; ++p)
        for (int w = 0; w < W; ++w) {
            x[p * W + w] = junk * (p + 5) ^ (junk >> w);
            y[p * W + w] = junk * (p + 9) ^ (junk << w);
            for (int i = 0; i < 32; ++i) {
                const size_t k = 32 * w + i;
                if (k < a.size()) x[p * W + w] = (x[p * W + w] & ~(1u << i)) | ((uint32_t)(a[k] >> p & 1) << i);
                if (k < b.size()) y[p * W + w] = (y[p * W + w] & ~(1u << i)) | ((uint32_t)(b[k] >> p & 1) << i);
            }
        }
    const int r = idb_lv_equal_length<NP, W, T>(x, y, (int)a.size(), t);
    ++asked;
    decided += r != 2;
    if (r != 2 && r != (d <= t))
        if (++fails < 6) std::printf("equal NP %d W %d T %d t %d: %zu lev %d got %d\n", NP, W, T, t, a.size(), d, r);
}

template <int NP, int W>
static void all_t(const std::string &a, const std::string &b, uint32_t junk)
{
    const int d = lev(a, b), dl = std::abs((int)a.size() - (int)b.size());
    if (dl <= 0) {
        one<NP, W, 1>(a, b, 0, d, junk);
        equal<NP, W, 1>(a, b, 0, d, junk);
        equal<NP, W, 1>(a, b, 1, d, junk);
        equal<NP, W, 2>(a, b, 2, d, junk);
        equal<NP, W, 3>(a, b, 3, d, junk);
        equal<NP, W, 4>(a, b, 4, d, junk);
    }
    if (dl <= 1) one<NP, W, 1>(a, b, 1, d, junk);
    if (dl <= 2) one<NP, W, 2>(a, b, 2, d, junk);
    if (dl <= 3) one<NP, W, 3>(a, b, 3, d, junk);
    if (dl <= 4) one<NP, W, 4>(a, b, 4, d, junk);
}

template <int NP, int W>
static void random_pairs(std::mt19937 &rng, int n)
{
    const int K = 1 << NP;
    for (int r = 0; r < n; ++r) {
        const int edge = 32 * (1 + (int)(rng() % W));
        const int L = rng() % 3 ? std::max(0, edge - (int)(rng() % 5)) : (int)(rng() % (32 * W + 1));
        const int k = rng() % 2 ? K : 2;  // two letters: many near ties
        std::string a, b;
        for (int i = 0; i < L; ++i) a.push_back((char)(rng() % k));
        b = a;
        for (int e = rng() % 8; e > 0; --e) {
            const int kind = rng() % 3;
            const size_t p = b.empty() ? 0 : rng() % b.size();
            if (kind == 0 && !b.empty()) b[p] = (char)(rng() % k);
            else if (kind == 1 && (int)b.size() < 32 * W) b.insert(b.begin() + (b.empty() ? 0 : rng() % (b.size() + 1)), (char)(rng() % k));
            else if (!b.empty()) b.erase(b.begin() + p);
        }
        all_t<NP, W>(a, b, rng());
        all_t<NP, W>(b, a, rng());
    }
}

int main()
{
    std::mt19937 rng(3);
    // every pair of strings of up to 6 letters over two, up to 4 over three
    std::vector<std::string> s2{""}, s3{""};
    for (size_t k = 0; s2[k].size() < 6; ++k)
        for (char c = 0; c < 2; ++c) s2.push_back(s2[k] + c);
    for (size_t k = 0; s3[k].size() < 4; ++k)
        for (char c = 0; c < 3; ++c) s3.push_back(s3[k] + c);
    for (auto *s : {&s2, &s3})
        for (auto &a : *s)
            for (auto &b : *s) {
                all_t<2, 1>(a, b, 0x9E3779B9u);
                all_t<5, 1>(a, b, 0x85EBCA6Bu);
            }
    random_pairs<5, 1>(rng, 20000);
    random_pairs<2, 1>(rng, 10000);
    random_pairs<2, 2>(rng, 10000);
    random_pairs<2, 3>(rng, 10000);
    random_pairs<2, 5>(rng, 6000);
    random_pairs<2, 8>(rng, 3000);
    std::printf("%ld checks, %ld of %ld equal-length ones decided early, %ld failed\n", checked, decided, asked, fails);
    return fails ? 1 : 0;
}
