// Counts flight steps of electrons that stand at t_sync already and do not leave
// the electron, the field gain and the escape flag as they are, over field cases.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstring>
#include <vector>
#include "../../loki-mc_amd/csrc/device_physics.h"
using namespace ekmc;

static uint64_t g_state = 88172645463325252ull;
static double u() {
    g_state ^= g_state << 13; g_state ^= g_state >> 7; g_state ^= g_state << 17;
    return (double)(g_state >> 11) * (1.0 / 9007199254740992.0);
}

template <typename V, int FC> static long run(int fieldCase, long& n) {
    CondParams c = {};
    c.fieldCase = fieldCase;
    const double E = 3000.0, B = 2e9;
    c.E[0] = E; c.E[2] = 0.5 * E;
    for (int k = 0; k < 3; ++k) { c.accel[k] = -kCharge / kMass * c.E[k]; c.fA[k] = (float)c.accel[k]; }
    c.cyclotron = B; c.cycRec = reciprocal(B);
    c.omega = fieldCase == FIELD_ECR ? B : 3.1e8; c.freq = c.omega / (2.0 * kPi);
    c.vEx = kCharge * c.E[0] / (kMass * B); c.az = kCharge * c.E[2] / kMass;
    c.fE0 = (float)c.E[0]; c.fE2 = (float)c.E[2]; c.fW = (float)B; c.fInvW = (float)(1.0 / B); c.fvEx = (float)c.vEx;
    c.fAz = (float)c.az; c.fEmw = (float)(kCharge / (kMass * c.omega)); c.fInvOmega = (float)(1.0 / c.omega);
    c.I = 100; c.N = 3e22; c.nRec = reciprocal(c.N); c.trial = 1e10; c.trialInv = 1e-10; c.trialRec = reciprocal(c.trial);
    c.step = 1.0; c.stepRec = reciprocal(c.step); c.tsync = 3.7e-7; c.envShift = 0;
    std::vector<V> nutot(c.I, (V)5e9), env(2 * kEnvBins, (V)5e9);
    DevProcesses pr = {};
    long bad = 0;
    for (int k = 0; k < 20000; ++k, ++n) {
        Electron<V> e;
        std::memset((void*)&e, 0, sizeof e);
        e.x = u() * 1e-3; e.y = -u() * 1e-3; e.z = u() * 1e-3; e.t = c.tsync;
        e.vx = (V)((u() - 0.5) * 2e6); e.vy = (V)((u() - 0.5) * 2e6); e.vz = (V)((u() - 0.5) * 2e6);
        // the energy an ionization leaves: shared, not worked out from the velocity
        e.eps = (V)((double)energy_of(e.vx, e.vy, e.vz) * (1.0 + 1e-7 * (u() - 0.5)));
        e.tfree = k & 1 ? (V)kNonDef : (V)(u() * 1e-10);
        e.nue = (V)9e9; e.stream = (uint64_t)k; e.event = 3;
        Electron<V> was;
        std::memcpy((void*)&was, (void*)&e, sizeof e);
        EventRng<V> rng(17, e.stream, e.event);
        double gain = 0;
        bool escape = false;
        const int st = step_a<V, FC, false>(c, pr, nutot.data(), env.data(), env.data() + kEnvBins, e, rng, escape, gain);
        if (st != STEP_DONE || escape || gain != 0 || std::memcmp(&was, &e, sizeof e) != 0) ++bad;
    }
    return bad;
}

int main() {
    long n = 0, bad = 0;
#define CASE(FC, field)                                                                                   \
    {                                                                                                     \
        const long b64 = run<double, FC>(field, n), b32 = run<float, FC>(field, n);                       \
        if (b64 || b32) std::printf(#FC " " #field ": %ld FP64, %ld FP32\n", b64, b32);                   \
        bad += b64 + b32;                                                                                 \
    }
    CASE(FIELD_DC, FIELD_DC)
    CASE(FIELD_AC, FIELD_AC)
    CASE(FIELD_DC_B, FIELD_DC_B)
    CASE(FIELD_ECR, FIELD_ECR)
    CASE(FIELD_AC_B, FIELD_AC_B)
    CASE(FLIGHT_DC_ANY, FIELD_DC)
    CASE(FLIGHT_DC_ANY, FIELD_DC_B)
    std::printf("%ld %ld\n", bad, n);
    return bad != 0;
}
