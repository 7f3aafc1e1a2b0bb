// How the integer trainers that are resident on the device (orbit_train.inc) are dealt to its blocks, and how many images a launch takes.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

constexpr uint32_t kSymWaves = 8;                         // of a resident block
constexpr uint32_t kSymGroupMax = 256;                    // images of a launch group
constexpr uint32_t kOrbTrainWorkers = 7;                  // waves that hold weights; the last wave exchanges words
constexpr uint32_t kOrbTrainMaxNit = 10;                  // orbits of a thread (six where a block holds three or four neurons)
constexpr uint32_t kOrbTrainAllNit = 6;                   // ... up to which all orbits are taken for reached
constexpr uint32_t kOrbTrainSplits = 8;                   // (a row of 16 lanes reads a neuron's words of that many blocks)
// Bytes of a group's operand, an image's planes and all, stay below: k_train_orbit_resident counts them in 32 bits and sends requests that
// it does not want to this offset, past the end.
constexpr size_t kOrbTrainOperand = (size_t)1 << 31;

// How a trainer's neurons and an image's rows are dealt to the blocks.
struct OrbitTrainPlan {
    uint32_t npb = 0, splits = 1, abreast = 1, tpw = 1, nit = 1, reached = 0;      // tpw: tiles of a wave side by side; orbits with an operand
    size_t lds = 0;
};

// Bytes between two neurons' rows in LDS: whole chunks of 64 orbits, so that a block's chunks follow each other.
constexpr uint32_t orbit_train_row(uint32_t orbits) { return (orbits + 63) / 64 * 512; }
// Bits of a neuron's number inside its block, below the distance in a block's word.
constexpr uint32_t orbit_train_bits(uint32_t npb) { return npb > 2 ? 2 : npb - 1; }
inline size_t orbit_train_lds(uint32_t npb, uint32_t orbits, uint32_t reached, bool u16, uint32_t N, uint32_t tpw)
{
    const size_t columns = npb > 2 ? 2 : 1;
    return (size_t)orbit_train_row(reached) * npb * (u16 ? 2 : 1) + orbit_train_row(orbits) + (size_t)kSymWaves * tpw * columns * (u16 ? 3 : 1) * 1024 + (size_t)npb * N * sizeof(float);
}

// K-steps of 64 of an operand row, an even number.
constexpr uint32_t orbit_train_steps(uint32_t reached) { return (reached * 8 + 127) / 128 * 2; }
// Bytes of an image's operand: fragments of 16 rows.
constexpr size_t orbit_train_operand(uint32_t nrr, uint32_t KS, bool u16) { return (size_t)(u16 ? 2 : 1) * ((nrr + 15) / 16) * KS * 1024; }

// How many neurons a block of a resident integer trainer holds and between how many blocks the rows are shared out: what is expected to
// take least.  In clocks of an image: a block's rows through its CU's 64 bytes a clock, its waves' instructions or the matrix pipes; a round of
// tiles, whose shares of k meet in the LDS; an update of 64 orbits a wave; two column tiles of uint16; the words of the blocks that hold the
// same neurons.  Fitted to every plan of 116 shapes (1 to 1024 neurons of 36 to 8281 elements, 40 to 720 rotations), up to four times apart:
// the plan taken is 0.3 % slower than the fastest in the mean, most with 256 uint8 neurons of 2025 elements (6.2 %).  npb 0: no way to hold the
// neurons.
inline OrbitTrainPlan plan_orbit_train(uint32_t N, uint32_t E, uint32_t orbits, uint32_t reached, uint32_t nrr, bool u16, uint32_t units, size_t lds_max)
{
    const uint32_t RT = (nrr + 15) / 16, planes = u16 ? 2 : 1, accs = u16 ? 3 : 1, products = u16 ? 4 : 1;
    const double most = (double)E * (u16 ? 65535.0 * 65535.0 : 255.0 * 255.0);
    OrbitTrainPlan best;
    double best_cost = 0.0;
    for (uint32_t npb = 1; npb <= 4; ++npb) {
        const uint32_t groups = (N + npb - 1) / npb, columns = npb > 2 ? 2 : 1, nit = (npb * ((orbits + 63) / 64) + kOrbTrainWorkers - 1) / kOrbTrainWorkers;
        const uint32_t streamed = nit > kOrbTrainAllNit ? reached : orbits, KS = orbit_train_steps(streamed);
        if (nit > (npb > 2 ? kOrbTrainAllNit : kOrbTrainMaxNit) || most >= (double)(1ull << (48 - orbit_train_bits(npb)))) break;
        if (orbit_train_operand(nrr, KS, u16) >= kOrbTrainOperand) continue;       // (a group of one image: see resident_group)
        uint32_t tiles_before = 0;
        for (uint32_t splits = 1; splits <= std::min(kOrbTrainSplits, RT) && groups * splits <= units; ++splits) {
            const uint32_t tiles = (RT + splits - 1) / splits;
            if (tiles == tiles_before) continue;
            // (More than six orbits a thread: rows that a compute unit takes longer to pull through than the orbits' product takes for an image.  Us an
            // image with everything, resident | image by image, neurons of 181 x 181 and images of 256 x 256 pixels, by tiles x KS x planes: 1048, 60
            // and 100 uint8 neurons 44.7 | 46.3 and 41.5 | 43.4, 60 uint16 39.0 | 49.1; 1572, 100 and 200 uint8 52.6 | 52.3 and 44.6 | 43.6; 2096, 100 uint8
            // 74.8 | 62.0, 60 and 100 uint16 61.2 | 60.1 and 49.6 | 52.4; 3144, 100 and 200 uint8 89.1 | 82.3 and 75.8 | 62.9, 100 uint16 77.5 | 69.3.)
            if (nit > kOrbTrainAllNit && tiles * KS * planes > 1600) continue;
            tiles_before = tiles;
            for (uint32_t abreast = 1; abreast <= 8; abreast *= 2)
                for (uint32_t tpw = 1; tpw <= (u16 ? 1u : 3u); tpw += 2) {
                    const size_t lds = orbit_train_lds(npb, orbits, streamed, u16, N, tpw);
                    if (lds + 2048 > lds_max) continue;
                    const uint32_t rounds = (tiles + abreast * tpw - 1) / (abreast * tpw), shares = kSymWaves / abreast;
                    const double stream = rounds * abreast * tpw * 16.0 * KS * planes;
                    const double issue = rounds * (KS / 2.0 / shares) * (columns * planes * 10.0 + tpw * planes * 4.0 + tpw * columns * products * 2.0 + 10.0) * 8.6;
                    const double matrix = rounds * abreast * tpw * (double)columns * KS * products * 4.0;
                    const double cost = (u16 ? 1.24 : 1.155) * std::max({stream, issue, matrix}) + rounds * (2850.0 + 110.0 * tpw * columns * accs + 10.0 * accs * shares * ((abreast * tpw * columns + 7) / 8)) +
                                        nit * (u16 ? 2070.0 : 1594.0) + (npb - 1) * (u16 ? 100.0 : 200.0) + (u16 && npb > 2 ? 1400.0 : 0.0) + (splits > 1 ? 100.0 + 300.0 * splits : 0.0) + (u16 ? 75.0 : 175.0) * (abreast - 1) + 3.0 * groups * splits;
                    if (!best.npb || cost < best_cost) {
                        best.npb = npb; best.splits = splits; best.abreast = abreast; best.tpw = tpw; best.nit = nit; best.lds = lds; best.reached = streamed;
                        best_cost = cost;
                    }
                }
        }
    }
    return best;
}

// Images of a launch group.  What one launch writes and the next reads (operand and values of an image: op_image and x_image bytes) stays within
// the last-level cache, down to eight images, and below kOrbTrainOperand, whatever that leaves (8 images of 16384 base rotations of 2080 orbits,
// uint16, would be 4.4e9 bytes).
inline uint32_t resident_group(uint32_t max_batch, size_t op_image, size_t x_image)
{
    size_t b = max_batch ? std::min(max_batch, kSymGroupMax) : kSymGroupMax;
    while (b > 8 && b * (op_image + x_image) > ((size_t)192 << 20)) --b;
    while (b > 1 && b * op_image >= kOrbTrainOperand) --b;
    return (uint32_t)b;
}
