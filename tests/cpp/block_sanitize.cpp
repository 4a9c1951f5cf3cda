// Test-only: a host driver that runs the block plan (lightsim2grid_amd/csrc/blocks.cpp) and its CPU replay
// (block_replay.cpp) on one grid, built with AddressSanitizer and UndefinedBehaviorSanitizer by
// tests/test_block_sanitize.py. Prints the tail's size and how many of its blocks the factor lacks, then "OK"
// (exit 0), or the first failed check (exit 1).
//
// Grid file (little-endian): int32 n, nnz; int32 Yp[n+1], Yi[nnz]; float64 Yx[2 nnz], Sbus[2 n],
// V0[2 n]; int32 nslack, slack_ids[nslack]; float64 slack_w[n]; int32 npv, pv[npv], npq, pq[npq]; more follows.
#include <cstdio>
#include <fstream>
#include <vector>

#include "../../lightsim2grid_amd/csrc/blocks.hpp"

extern "C" int block_replay_solve(int n, const int* Yp, const int* Yi, const double* Yx, const double* Sbus,
                                  const int* slack_ids, int nslack, const double* w, const int* pv, int npv,
                                  const int* pq, int npq, int single_slack, double* V, int max_iter, double tol, int G,
                                  int waves, int by_life, int* status, int* info);

namespace {

template <typename T>
std::vector<T> rd(std::ifstream& f, size_t k) {
    std::vector<T> v(k);
    if (k) f.read(reinterpret_cast<char*>(v.data()), (std::streamsize)(k * sizeof(T)));
    return v;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc < 3) return 2;
    std::ifstream f(argv[1], std::ios::binary);
    const bool solvable = argv[2][0] == '1';
    const auto head = rd<int>(f, 2);
    const int n = head[0], nnz = head[1];
    const auto Yp = rd<int>(f, n + 1), Yi = rd<int>(f, nnz);
    const auto Yx = rd<double>(f, 2 * (size_t)nnz), S = rd<double>(f, 2 * (size_t)n), V0 = rd<double>(f, 2 * (size_t)n);
    const auto slack = rd<int>(f, rd<int>(f, 1)[0]);
    const auto w = rd<double>(f, n);
    const auto pv = rd<int>(f, rd<int>(f, 1)[0]);
    const auto pq = rd<int>(f, rd<int>(f, 1)[0]);
    if (!f) return 2;
    int tail = 0, absent = 0;
    for (int single = slack.size() == 1 ? 1 : 0; single >= 0; --single) {
        pfgpu::YbusPattern Y;
        Y.n = n;
        Y.p = Yp;
        Y.i = Yi;
        const pfgpu::JPattern J = pfgpu::build_jacobian_pattern(Y, slack.data(), (int)slack.size(), w.data(), pv.data(),
                                                                (int)pv.size(), pq.data(), (int)pq.size(), single != 0);
        const pfgpu::BlockPlan P = pfgpu::build_block_plan(Y, J, pfgpu::column_order(J));
        for (int x : P.tail_src) {
            if (x < 0 || x >= 2 * P.npairs) return std::printf("a tail number lies outside the values: %d\n", x), 1;
            absent += x / 2 == P.zpair;
        }
        tail += P.m;
        const pfgpu::BlockPlan L = pfgpu::by_life(P);
        for (int G : {1, 4, 32})
            for (int waves : {4, 16})
                for (int nlds : {P.fixed_pairs, P.npairs}) (void)pfgpu::build_block_streams(P, G, waves, 4, nlds);
        (void)pfgpu::build_block_streams(L, 1, 16, 8, L.npairs);
        if (!solvable) continue;
        for (int life : {0, 1}) {
            std::vector<double> V = V0;
            int status = -1, info[6];
            const int it = block_replay_solve(n, Yp.data(), Yi.data(), Yx.data(), S.data(), slack.data(),
                                              (int)slack.size(), w.data(), pv.data(), (int)pv.size(), pq.data(),
                                              (int)pq.size(), single, V.data(), 10, 1e-8, 1, 16, life, &status, info);
            if (it < 0 || status != 0 || info[5] != 0)
                return std::printf("replay: iterations %d status %d conflicts %d\n", it, status, info[5]), 1;
        }
    }
    std::printf("tail %d absent %d OK\n", tail, absent);
    return 0;
}
