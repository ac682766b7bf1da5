// Storage for the CPU execution shim's per-launch state.  Test infrastructure only.
#define TAH_EMU_IMPL
#include <hip/hip_runtime.h>

extern "C" void tah_emu_run_blocks(unsigned first, unsigned count) {
    emu::g_first_block = first;
    emu::g_block_count = count;
    emu::g_ors.clear();
}
extern "C" int tah_emu_ors(const void** at, int n) {  // returns how many there were
    for (int i = 0; i < n && i < (int)emu::g_ors.size(); ++i) at[i] = emu::g_ors[i];
    return (int)emu::g_ors.size();
}
