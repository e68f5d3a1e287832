// Checks of once_per_device.h, one bit of the result each; 0: all hold.
#include "once_per_device.h"

extern "C" int opd_check() {
    slai::OncePerDevice once;
    int calls = 0, status = 0, bad = 0;
    const auto at = [&](int device) { return once(device, [&] { ++calls; return status; }); };
    status = 7;
    if (at(0) != 7 || calls != 1) bad |= 1;                    // a failure is reported
    status = 0;
    if (at(0) != 0 || calls != 2) bad |= 2;                    // ... and tried again
    if (at(0) != 0 || calls != 2) bad |= 4;                    // set once
    if (at(1) != 0 || calls != 3) bad |= 8;                    // another device of the same process
    if (at(63) != 0 || at(63) != 0 || calls != 4) bad |= 16;
    if (at(64) != 0 || at(64) != 0 || calls != 6) bad |= 32;   // beyond what is remembered: each time
    return bad;
}
