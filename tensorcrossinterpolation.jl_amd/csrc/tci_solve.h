// tci_solve.h — the kernels of tci_solve.hip, by threads per solve.
//
// tci_solve.hip is compiled once per team (TCI_SOLVE_TEAM), as an object of its own:
// the engine with the register tiles takes the compiler 10 to 20 s for each functor,
// and one object of all of them took 155 s while make had nothing to run beside it.
#pragma once

namespace tci {

// the solve kernel for a functor kind (0: mixed kinds)
const void *solve_kernel_64(int fkind);
const void *solve_kernel_256(int fkind);
const void *solve_kernel_512(int fkind);
const void *solve_kernel_1024(int fkind);
// the serving kernel
const void *serve_kernel_256();
const void *serve_kernel_512();

}  // namespace tci
