// mci_rtc.hpp — the caller's device functors (MCI_PDF_DEVICE, MCI_OBS_DEVICE): the generic step
// kernels (mci_step_kernels.hpp) built at run time together with the functors' sources.
#pragma once

#include "mci_kernels.hpp"

#include <string>
#include <vector>

namespace mcid
{
// a functor's name (its functions are NAME_proto, ... or NAME_observable) and source
struct RtcFunctor
{
    std::string name, source;
};

// the generic step kernels of one program (loaded on one device), by StateKind.  Each kind is a build of its
// own: a program is built in the kinds its chain takes.
struct RtcKernels
{
    hipFunction_t sample[STATE_KINDS] = {}, calibrate[STATE_KINDS] = {};
    bool any() const { return kinds() != 0; }
    bool has(int k) const { return (kinds() & k) == k; }
    int kinds() const
    {
        int k = 0;
        for (int i = 0; i < STATE_KINDS; ++i) { k |= sample[i] ? 1 << i : 0; }
        return k;
    }
};

// true when name is a C identifier
bool rtc_valid_name(const std::string &name);
// the program text: the functors' sources (one copy per name), their dispatch by index (pdfs[i] is
// sampling function index i, obs[i] observable index i; the move, if any), then the step kernels.
// Returns false with a message when two functors share a name but not a source.
// move: the caller's trial move (or null)
bool rtc_program(const std::vector<RtcFunctor> &pdfs, const std::vector<RtcFunctor> &obs, const RtcFunctor *move, std::string &text,
                 std::string &msg);
// compiles text for arch (e.g. "gfx950") without loading it; log: the compiler's messages.  One kind: the
// functors are the same text in both.
int rtc_check(const std::string &text, const char *arch, std::string &log);
// the kernels of text on the current device, those of the given kinds (bits 1 << StateKind) among
// them: compiled and loaded once per text, device and kind
int rtc_get(const std::string &text, int kinds, RtcKernels &out, std::string &log);
hipError_t rtc_launch_sample(const RtcKernels &k, const Chain &c, int64_t nsteps, int acc, const uint8_t *active, hipStream_t s,
                             const CalibCtrl *skip);
hipError_t rtc_launch_calibrate_indep(const RtcKernels &k, const Chain &c, int nfind, double target, int64_t min_stat,
                                      const double *dimSizes, hipStream_t s);
} // namespace mcid
