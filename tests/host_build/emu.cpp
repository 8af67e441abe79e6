// The switch between a workgroup's scheduler and its lanes (x86-64): callee-saved
// registers on the old stack, then the new stack's.
#if !defined(__x86_64__)
#error "the host build switches stacks with x86-64 code"
#endif
__asm__(
    ".text\n.globl emu_switch\n.type emu_switch,@function\n"
    "emu_switch:\n"
    "  pushq %rbp\n  pushq %rbx\n  pushq %r12\n  pushq %r13\n  pushq %r14\n  pushq %r15\n"
    "  movq %rsp, (%rdi)\n  movq %rsi, %rsp\n"
    "  popq %r15\n  popq %r14\n  popq %r13\n  popq %r12\n  popq %rbx\n  popq %rbp\n"
    "  ret\n"
    ".size emu_switch,.-emu_switch\n"
    ".section .note.GNU-stack,\"\",@progbits\n");
