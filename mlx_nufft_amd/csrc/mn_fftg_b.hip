// Line lengths of the general pruned FFT, every sixth of the table (the files
// only divide the compile time).
#include "mn_fftg.h"

namespace mn {

const FgEntry *fg_entries_b(int *count) {
    static const FgEntry table[] = {
        fg::entry<6>(), fg::entry<16>(), fg::entry<30>(), fg::entry<50>(), fg::entry<80>(),
        fg::entry<120>(), fg::entry<160>(), fg::entry<225>(), fg::entry<288>(),
        fg::entry<384>(), fg::entry<486>(), fg::entry<625>(), fg::entry<750>(),
        fg::entry<960>(), fg::entry<1152>(), fg::entry<1350>(), fg::entry<1620>(),
        fg::entry<2000>()};
    *count = (int)(sizeof(table) / sizeof(table[0]));
    return table;
}

}  // namespace mn
