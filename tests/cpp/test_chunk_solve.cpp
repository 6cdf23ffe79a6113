// The chunked line solve of the fused sweeps on the CPU, from the tables the
// kernels read (chunk_table), for every line length 16..512 that a fused axis
// can have: chunks of 8 and 16 points, equal, one short or balanced ones;
// derivative tables of closure and seam ends, filter tables of closure and
// cyclic lines.  Checks that the chunks cover the line, and the solution
// (carries cut off at carry_reach, as the kernels fold them) against the
// unchunked recurrences in long double.
#include "sweep_parts.hpp"

#include <cmath>
#include <cstdio>

using namespace cs;
using namespace cs::fused;

static double rnd(unsigned& x) {
    x = x * 1664525u + 1013904223u;
    return (double)(x >> 8) / (1 << 24) - 0.5;
}

int main() {
    double worst = 0.0;
    int lines = 0;
    for (int K : {8, 16})
        for (int n = 16; n <= 512; n++)
            for (int op : {OP_DERIV, OP_FILTER})
                for (int seam : {0, 1}) {
                    const int P = (n + K - 1) / K, NP = P * K;
                    int covered = 0, shortest = K, longest = 0;
                    for (int c = 0; c < P; c++) {
                        const int s = chunk_start(n, P, K, c), L = chunk_start(n, P, K, c + 1) - s;
                        if (s != covered) { std::printf("n=%d K=%d chunk %d starts at %d\n", n, K, c, s); return 1; }
                        covered += L;
                        shortest = L < shortest ? L : shortest;
                        longest = L > longest ? L : longest;
                    }
                    const bool fits = chunks_fit(n, P, K);
                    const int first = chunk_start(n, P, K, 1), last = n - chunk_start(n, P, K, P - 1);
                    if (covered != n || longest > K || shortest < 4 ||
                        (fits && (shortest < K - 1 || first != K || last != K))) {
                        std::printf("n=%d K=%d: chunks of %d..%d rows, %d covered\n", n, K, shortest, longest, covered);
                        return 1;
                    }
                    std::vector<double> h, t;
                    if (build_line_table(op, n, seam, seam, 0.49, K, h)) return 1;
                    chunk_table(h, n, K, P, t);
                    unsigned seed = (unsigned)(n * 7 + K + op * 3 + seam);
                    std::vector<double> f(n), r(NP, 0.0), G(P, 0.0), X(P, 0.0), cf(P), cb(P);
                    for (double& v : f) v = rnd(seed);
                    // the recurrences of the whole line, long double
                    std::vector<long double> x(n);
                    long double g = 0.0L;
                    for (int j = 0; j < n; j++) x[j] = g = (long double)h[j] * f[j] + (long double)h[n + j] * g;
                    for (int j = n - 2; j >= 0; j--) x[j] += (long double)h[2 * n + j] * x[j + 1];
                    // chunk by chunk
                    const int reach = op == OP_FILTER ? P : kCarryRows / K;
                    for (int c = 0; c < P; c++) {
                        const int s = chunk_start(n, P, K, c), L = chunk_start(n, P, K, c + 1) - s;
                        for (int i = 0; i < L; i++) r[c * K + i] = f[s + i];
                        double p = 0.0;
                        for (int i = 0; i < K; i++) {
                            const int o = c * K + i;
                            r[o] = p = std::fma(t[o], r[o], t[NP + o] * p);
                        }
                        cf[c] = p;
                    }
                    for (int c = 0; c < P; c++)
                        for (int b = c - reach > 0 ? c - reach : 0; b < c; b++)
                            G[c] = std::fma(t[3 * NP + b * K + K - 1], G[c], cf[b]);
                    for (int c = 0; c < P; c++) {
                        const int L = chunk_start(n, P, K, c + 1) - chunk_start(n, P, K, c);
                        double p = 0.0;
                        for (int i = 0; i < K; i++) {
                            const int o = c * K + i;
                            r[o] = i < L ? std::fma(t[3 * NP + o], G[c], r[o]) : 0.0;
                        }
                        for (int i = K - 1; i >= 0; i--) {
                            const int o = c * K + i;
                            r[o] = p = std::fma(t[2 * NP + o], p, r[o]);
                        }
                        cb[c] = p;
                    }
                    for (int c = 0; c < P; c++)
                        for (int b = c + reach < P - 1 ? c + reach : P - 1; b > c; b--)
                            X[c] = std::fma(t[4 * NP + b * K], X[c], cb[b]);
                    double err = 0.0, big = 0.0;
                    for (int c = 0; c < P; c++) {
                        const int s = chunk_start(n, P, K, c), L = chunk_start(n, P, K, c + 1) - s;
                        for (int i = 0; i < L; i++) {
                            const double v = std::fma(t[4 * NP + c * K + i], X[c], r[c * K + i]);
                            err = std::fmax(err, (double)fabsl(x[s + i] - v));
                            big = std::fmax(big, (double)fabsl(x[s + i]));
                            if (op == OP_FILTER && seam && t[5 * NP + c * K + i] != h[5 * n + s + i]) return 1;
                        }
                    }
                    worst = std::fmax(worst, err / big);
                    lines++;
                }
    std::printf("%d lines, largest relative error %.2e\n", lines, worst);
    // a few units of 2^-53 a row, amplified by at most the filter factors' 1/(1 - 0.82)
    return worst < 64 * 1.1e-16 ? 0 : 1;
}
