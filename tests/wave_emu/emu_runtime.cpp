// State of the CPU execution shim (tests/wave_emu/hip_cpu.hpp).  TEST INFRASTRUCTURE ONLY.
#include "hip_cpu.hpp"

#include <cstdlib>

// launches run at once on the CPU: no graph capture (hip_cpu.hpp)
static const int g_no_graphs = setenv("MI_GRAPHS", "0", 1);

// the device's fast log2 (declared by the C library's math header, not
// exported by it); only the scorer features use it
#include <cmath>
extern "C" float __log2f(float x) noexcept { return log2f(x); }

namespace emu {
EMU_LANE_LOCAL Ctx* g = nullptr;
EMU_LANE_LOCAL int lane = 0;
EMU_LANE_LOCAL const void* t_kernarg = nullptr;
EMU_LANE_LOCAL dim3 t_block, t_thread;
dim3 g_bdim, g_gdim;
YieldBarrier* g_blockbar = nullptr;

#ifdef MI_EMU_FIBERS
// The lanes as fibers: a waiting lane switches to the next one that is not done.
extern "C" void emu_switch(void** save, void* to);   // the callee-saved registers of the System V ABI
asm(R"(
.globl emu_switch
emu_switch:
  pushq %rbp; pushq %rbx; pushq %r12; pushq %r13; pushq %r14; pushq %r15
  movq %rsp, (%rdi)
  movq %rsi, %rsp
  popq %r15; popq %r14; popq %r13; popq %r12; popq %rbx; popq %rbp
  ret
)");
struct Fiber {
    void* sp = nullptr;
    bool done = false;
    const void* kernarg = nullptr;
    dim3 block;
};
static std::vector<Fiber> fibers;
static std::vector<std::unique_ptr<char[]>> stacks;
static unsigned cur;
static void* launcher;
static const std::function<void(unsigned)>*fiber_set, *fiber_work;

void lane_yield()
{
    const unsigned c = cur, nt = (unsigned)fibers.size();
    unsigned n = c;
    do n = n + 1 == nt ? 0 : n + 1;
    while (fibers[n].done && n != c);
    fibers[c].kernarg = t_kernarg;
    fibers[c].block = t_block;
    void* to = fibers[n].sp;
    if (fibers[n].done) to = launcher;   // every fiber is
    else if (n == c) return;
    else {
        cur = n;
        (*fiber_set)(n);
        t_kernarg = fibers[n].kernarg;
        t_block = fibers[n].block;
    }
    emu_switch(&fibers[c].sp, to);
}

static void fiber_entry()
{
    (*fiber_work)(cur);
    fibers[cur].done = true;
    lane_yield();
    abort();
}

void run_fibers(unsigned nt, const std::function<void(unsigned)>& set, const std::function<void(unsigned)>& work)
{
    const size_t size = 1 << 18;
    fiber_set = &set;
    fiber_work = &work;
    while (stacks.size() < nt) stacks.emplace_back(new char[size]);
    fibers.assign(nt, Fiber{});
    for (unsigned i = 0; i < nt; i++) {
        void** sp = (void**)(((uintptr_t)stacks[i].get() + size) & ~(uintptr_t)15);
        *--sp = nullptr;   // the entry's return address: never used
        *--sp = (void*)fiber_entry;
        for (int q = 0; q < 6; q++) *--sp = nullptr;
        fibers[i].sp = sp;
    }
    cur = 0;
    set(0);
    emu_switch(&launcher, fibers[0].sp);
}
#endif
}  // namespace emu
