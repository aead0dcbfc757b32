// Counts, over energies and variates at the ends of the samplers, elastic
// collisions that change the speed by more than the recoil, and ionizations whose
// electrons do not share the energy that is left.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <initializer_list>
#include "../../loki-mc_amd/csrc/device_physics.h"
using namespace ekmc;

constexpr double kTarget = 28.0 * 1.66053906660e-27;

template <typename V> static long run(int scat, double p0, double p1, bool ion, long& n) {
    ProcRec pc = {};
    pc.type = ion ? 1 : 0;
    pc.scat = scat;
    pc.params[0] = p0;
    pc.params[1] = p1;
    pc.tMass = kTarget;
    pc.rMass = kMass * kTarget / (kMass + kTarget);
    pc.energyLoss = ion ? 12.0 : 0.0;
    pc.wParam = 12.0;
    DevProcesses pr = {};
    pr.P = pr.G = 1;
    pr.proc = &pc;
    pr.ionizOp = 3;  // a uniform share
    const double ends[] = {0.0, std::ldexp(1.0, -24), 1e-3, 0.5, 1.0 - std::ldexp(1.0, -23), 1.0 - std::ldexp(1.0, -24)};
    // recoil of the target, and the roundings of a collision: the speed's square
    // and the three components of a unit vector, a few dozen units in the last place
    const double eps = sizeof(V) == 4 ? 64 * std::ldexp(1.0, -24) : 64 * std::ldexp(1.0, -53);
    const double lost = 4.0 * kMass * kTarget / ((kMass + kTarget) * (kMass + kTarget));
    long bad = 0;
    for (int k = 0; k < 400; ++k) {
        const double energy = (ion ? 12.001 : 1e-6) * std::pow(ion ? 40.0 : 1e9, k / 399.0);
        for (double r6 : ends)
            for (double r7 : {0.1, 0.6, 1.0}) {
                double tape[11];
                for (double& t : tape) t = 0.37;
                tape[6] = r6;
                tape[7] = r7;
                tape[9] = r6;
                const double speed = std::sqrt(2.0 * energy * kCharge / kMass);
                Electron<V> e = {};
                e.vx = (V)(0.48 * speed); e.vy = (V)(-0.6 * speed); e.vz = (V)(0.64 * speed);
                e.eps = energy_of(e.vx, e.vy, e.vz);
                const double was = (double)e.eps;
                EventRng<V> rng(0, 0, 0, tape);
                CollOut<V> o = {};
                const V Vt[3] = {(V)0, (V)0, (V)0};
                apply_collision<V, false>(pr, e, rng, o, 0, Vt, false);
                if (o.pid < 0) continue;
                ++n;
                double now = 0.5 * kMass * ((double)e.vx * e.vx + (double)e.vy * e.vy + (double)e.vz * e.vz) / kCharge;
                double low = was * (1.0 - lost), high = was;
                if (ion) {
                    now += 0.5 * kMass * ((double)o.ejv[0] * o.ejv[0] + (double)o.ejv[1] * o.ejv[1] + (double)o.ejv[2] * o.ejv[2]) / kCharge;
                    low = high = was - 12.0;
                }
                if (!(now >= low - eps * was && now <= high + eps * was)) ++bad;
            }
    }
    return bad;
}

int main() {
    // Surendra, screened Coulomb (energy before and after), forward, isotropic
    const double models[][3] = {{3, 0, 0}, {4, 0, 1.0}, {4, 1, 0.05}, {1, 0, 0}, {0, 0, 0}};
    long n = 0, bad = 0;
    for (const auto& m : models)
        for (int ion = 0; ion < 2; ++ion) {
            const long b64 = run<double>((int)m[0], m[1], m[2], ion != 0, n), b32 = run<float>((int)m[0], m[1], m[2], ion != 0, n);
            if (b64 || b32) std::printf("model %d ion %d: %ld FP64, %ld FP32\n", (int)m[0], ion, b64, b32);
            bad += b64 + b32;
        }
    std::printf("%ld %ld\n", bad, n);
    return bad != 0;
}
