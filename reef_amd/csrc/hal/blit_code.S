// The copy kernel's code object, as built from blit.hip.
    .section .rodata
    .balign 4096
    .globl reef_blit_code
reef_blit_code:
    .incbin "build/reef_blit.elf"
    .globl reef_blit_code_end
reef_blit_code_end:
    .byte 0
    .section .note.GNU-stack,"",@progbits
