// dbx_sweeps.h -- when the level sweeps of a world or an island overlap on several waves.
// Plain constant expressions, for the kernels and for a compiler without HIP.
#pragma once

namespace dbx {

// The waves publish their progress as an int: sweep * levels + levels done, and the start
// of a wave's next sweep, (sweep + waves) * levels, when one ends.  A count past 2^31 would
// let a level pass before the one it waits for, or wait for ever; such sweeps run one
// after the other instead (it takes hours to run as many levels).
constexpr bool sweeps_countable(long long sweeps, int waves, int levels) {
    return (sweeps + waves + 1) * ((long long)levels + 1) < (1ll << 30);
}

// Whether `sweeps` sweeps gain at least a tenth by overlapping on `waves` waves: a sweep
// starts at least lag levels after the one before it, and after the one `waves` before it
// on the same wave has ended.
constexpr bool overlap_gains(long long sweeps, int waves, int lag, int levels) {
    const long long turn = (levels + waves - 1) / waves, stride = lag > turn ? lag : turn;
    return 10 * ((sweeps - 1) * stride + levels) <= 9 * sweeps * levels;
}

// Waves, at most `most`, of the sweeps of a big island whose impulses lie in global memory
// (velocity_sweep_far); 0: one after the other.
constexpr int far_waves(long long sweeps, int most, int lag, int levels, bool always) {
    if (sweeps < 2 || levels < 2 || !sweeps_countable(sweeps, most, levels)) return 0;
    const int useful = (levels + lag - 1) / lag, waves = always || useful > most ? most : useful;
    return waves > 1 && (always || overlap_gains(sweeps, waves, lag, levels)) ? waves : 0;
}

} // namespace dbx
