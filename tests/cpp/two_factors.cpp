// Two DIC factorisations on one mesh, then a smoothing sweep with the first: the numbers are the first one's,
// whichever the mesh's one-launch plan last laid out (brae_amd/csrc/sweep.hpp), and the same sweep with the second,
// and with the first factored again, are theirs. Compared to the bit with the host loops on a chain-and-skip mesh of
// argv[1] cells. Prints "ok".
#include "../../brae_amd/csrc/mfv_internal.hpp"

#include <cstdio>
#include <cstdlib>
#include <random>

using namespace mfv;

namespace {

struct System
{
    std::vector<double> diag, upper, rD;
    DBuf<double> dDiag, dUpper, dRD;
    LduView view;
};

// psi + DIC(b - A psi), the host loops (gamg_solver_cpp.cu:194-231, 277-293)
std::vector<double> hostSmooth(const Mesh& m, const System& S, const std::vector<double>& b, std::vector<double> psi)
{
    const int n = m.nCells, nF = m.nFaces;
    std::vector<double> r(n), w(n);
    for (int c = 0; c < n; ++c) r[c] = b[c] - S.diag[c] * psi[c];
    // a cell's lower faces before its owned ones, as the residual takes them
    for (int f = 0; f < nF; ++f) r[m.hNeighbour[f]] -= S.upper[f] * psi[m.hOwner[f]];
    for (int f = 0; f < nF; ++f) r[m.hOwner[f]] -= S.upper[f] * psi[m.hNeighbour[f]];
    for (int c = 0; c < n; ++c) w[c] = S.rD[c] * r[c];
    for (int f = 0; f < nF; ++f) w[m.hNeighbour[f]] -= S.rD[m.hNeighbour[f]] * S.upper[f] * w[m.hOwner[f]];
    for (int f = nF - 1; f >= 0; --f) w[m.hOwner[f]] -= S.rD[m.hOwner[f]] * S.upper[f] * w[m.hNeighbour[f]];
    for (int c = 0; c < n; ++c) psi[c] += w[c];
    return psi;
}

} // namespace

int main(int argc, char** argv)
{
    const int n = argc > 1 ? std::atoi(argv[1]) : 1000;
    Ctx c;
    hipCheck(hipSetDevice(0), "device");
    hipCheck(hipStreamCreate(&c.stream), "stream");
    {
        std::vector<int> own, nei;
        for (int i = 0; i + 1 < n; ++i)
        {
            own.push_back(i);
            nei.push_back(i + 1);
            if (i % 3 == 0 && i + 17 < n)
            {
                own.push_back(i);
                nei.push_back(i + 17);
            }
        }
        Mesh m;
        buildMesh(c, m, n, (int)own.size(), own.data(), nei.data(), 0, nullptr);
        std::mt19937_64 rng(5);
        std::uniform_real_distribution<double> u(0.2, 1.0);
        std::vector<double> b(n), psi0(n);
        for (int i = 0; i < n; ++i)
        {
            b[i] = u(rng);
            psi0[i] = u(rng);
        }
        System S[2];
        for (System& s : S)
        {
            s.diag.assign(n, 0.1);
            s.upper.resize(own.size());
            for (size_t f = 0; f < own.size(); ++f)
            {
                s.upper[f] = -u(rng);
                s.diag[own[f]] -= s.upper[f];
                s.diag[nei[f]] -= s.upper[f];
            }
            s.rD = s.diag;
            for (size_t f = 0; f < own.size(); ++f) s.rD[nei[f]] -= s.upper[f] * s.upper[f] / s.rD[own[f]];
            for (double& v : s.rD) v = 1.0 / v;
            s.dDiag.upload(s.diag, c.stream);
            s.dUpper.upload(s.upper, c.stream);
            s.dRD.resize(n);
            s.view = LduView{n, (int)own.size(), s.dDiag.p, s.dUpper.p, s.dUpper.p};
        }
        DBuf<double> db, psi, rA, w;
        db.upload(b, c.stream);
        rA.resize(n);
        w.resize(n);
        auto check = [&](const char* what, const System& s, unsigned factor) {
            psi.upload(psi0, c.stream);
            launchDicSmooth(c, m, s.view, factor, s.dRD.p, db.p, psi.p, 1, rA.p, w.p);
            const std::vector<double> got = psi.download(c.stream), want = hostSmooth(m, s, b, psi0);
            for (int i = 0; i < n; ++i)
                if (got[i] != want[i])
                {
                    std::printf("%s: cell %d: %.17g, not %.17g\n", what, i, got[i], want[i]);
                    std::exit(1);
                }
        };
        const unsigned f0 = launchDicFactor(c, m, S[0].view, S[0].dRD.p);
        check("the first", S[0], f0);
        const unsigned f1 = launchDicFactor(c, m, S[1].view, S[1].dRD.p);
        check("the first, after the second was factored", S[0], f0);
        check("the second", S[1], f1);
        check("the first, factored again", S[0], launchDicFactor(c, m, S[0].view, S[0].dRD.p));
    }
    hipCheck(hipStreamDestroy(c.stream), "stream");
    std::puts("ok");
    return 0;
}
